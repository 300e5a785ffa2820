// gfx950 kernels of the AFAR SSP-RK3 stage pipeline.
//
// Per RK stage: reconstruct (cell) -> bvd (cell) -> flux (face) -> update
// (cell: residual gather + RK update + boundary ghosts); one CFL pass per
// step.  The kernels are templated on the reconstruction/flux type R: R =
// double is the all-FP64 transcription of the reference kernels, R = float is
// the mixed-precision path (state, residual and RK update stay FP64).
//
// Reference kernels: src/CUDA/cudaEuler2DmixO3RK3/cudaLimiter.h:35-464,
// cudaRiemannSolver.h:7-271, cudaFieldOperation.h:51-268,
// src/CUDA/BCs/2D/cudaEulerBCs.h:42-73, launch order GPUevolve.cu:207-306.
//
// Arithmetic is written operation-for-operation in the reference's order and
// the file is built with -ffp-contract=off, so the FP64 path reproduces the
// host oracle bit for bit.
#include <hip/hip_runtime.h>

#include "afar_math.h"
#include "kernels.h"

namespace afar {

// Thresholds of the reference (cudaLimiter.h:4-7), in the working type.
template <typename R> struct K {
    static constexpr R SMALL = (R)1e-5;
    static constexpr R VSMALL = (R)1e-10;
    static constexpr R BVD_FACTOR = (R)0.5;
    static constexpr R VALID_LIM_FACTOR = (R)0.9;
};

__device__ __forceinline__ size_t sell(int c, int k, int Kw) {
    return ((size_t)(c >> 6) * Kw + k) * 64 + (c & 63);
}

// Block -> tile mapping (TileMap): the tile of this block, or -1.
// Blocks are dispatched round-robin over the 8 XCDs, each with its own L2, and
// what one kernel leaves in an L2 the next one finds there if the same XCD
// works on the same cells.  Every kernel's tiles, whatever their size, are cut
// into the same number of chunks (cells and faces lie in Hilbert order, so a
// chunk is a compact region whose halos are mostly read through the same L2),
// and chunk j is XCD j % 8's.  With chunks of 32 blocks of each kernel, 64 or
// 256 cells a block, a cell's XCD changed from kernel to kernel: 20k quads 80.7
// -> 73.1 us a step, in FP32-mixed 69.2 -> 65.8, 17k periodic quads 64.3 ->
// 59.5, 134k triangles 170.6 -> 161.1, 48k in FP32-mixed 96.5 -> 89.9.
__device__ __forceinline__ int xcd_tile(const TileMap& m) {
    const unsigned b = blockIdx.x, i = b >> 3;
    const unsigned q = m.magic ? __umulhi(i, m.magic) : i;  // i / per
    const unsigned long long j = 8ull * q + (b & 7);        // the chunk
    const int lo = (int)((j * m.n) >> m.mlog), hi = (int)(((j + 1) * m.n) >> m.mlog);
    const int tile = lo + (int)(i - q * m.per);
    return tile < hi ? tile : -1;
}

// exp and erfc of KFVS, both sides of a face at once: the library's own
// functions (afar_math.h) in the working precision, which depend on no vendor
// math library, so the host restatements reproduce them bit for bit.  A wave
// with a shock face takes both flux branches, 21k cycles against 9k without
// one, most of them in these serial chains (eight exps, two series of 26
// terms): side by side, with the limiters' divisions (face_limiters), the
// pass takes 7.8 instead of 8.5 us on the 20k-cell corner, FP32-mixed 5.8
// instead of 6.2, and 116.6 instead of 118.6 on the 1.5M-cell Riemann problem.
__device__ __forceinline__ void erfc_exp(const double (&x)[2], const double (&a)[2], double (&c)[2], double (&e)[2]) {
    afar_erfc_exp_n<2>(x, a, c, e);
}
__device__ __forceinline__ void erfc_exp(const float (&x)[2], const float (&a)[2], float (&c)[2], float (&e)[2]) {
    afar_erfc_exp_nf<2>(x, a, c, e);
}

// ---------------------------------------------------------------- K3 least squares

template <typename R>
__global__ void k_lsq(DevPtrs<R> p) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= p.nc) return;
    const int C = p.ccnt[c];
    double Sxx = 0.0, Sxy = 0.0, Syy = 0.0;
    for (int i = 0; i < C; ++i) {
        const double2 e = p.slot_e[sell(c, i, p.maxC)];
        Sxx += e.x * e.x;
        Sxy += e.x * e.y;
        Syy += e.y * e.y;
    }
    for (int i = 0; i < C; ++i) {
        const double2 e = p.slot_e[sell(c, i, p.maxC)];
        typename VT<R>::v2 m;
        m.x = (R)((Syy * e.x - Sxy * e.y) / (Sxx * Syy - Sxy * Sxy));
        m.y = (R)((-Sxy * e.x + Sxx * e.y) / (Sxx * Syy - Sxy * Sxy));
        p.lsq[sell(c, i, p.maxC)] = m;
        // the centre distance K5 divides by (cudaLimiter.h:280), once here
        p.slot_dr[sell(c, i, p.maxC)] = (R)afar_hypot(e.x, e.y);
    }
}

// The gas as the face passes use it: what every face would divide out for
// itself is formed once on the host, with the kernels' expressions in the
// precision they use it in (a float widened to double comes back exactly).
struct GasArgs {
    double R, Cv, CFL;
    double gamma;  // (Cv + R) / Cv
    double c2T;    // (R / Cv + 1) R, the CFL bound's
    double Kd;     // KFVS: 2 Cv / R - 2
};
template <typename R> static inline GasArgs gas_args(double Rg, double Cv, double CFL) {
    return {Rg, Cv, CFL, (Cv + Rg) / Cv, (Rg / Cv + 1.0) * Rg, (double)((R)2 * (R)Cv / (R)Rg - (R)2)};
}

// ---------------------------------------------------------------- K4 time step

__device__ __forceinline__ double block_min_256(double v, double* wmin) {
    // wavefront min through cross-lane swizzles, then across the 4 waves
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off);
        v = o < v ? o : v;
    }
    if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = v;
    __syncthreads();
    double m = wmin[0];
    for (int w = 1; w < 4; ++w) m = wmin[w] < m ? wmin[w] : m;
    __syncthreads();
    return m;
}

// Time-step bound of one internal face (cudaFieldOperation.h:124-180).
// g: the distance of the two cell centres and the owner's share of it
// (DevPtrs::fcfl); c2T: sound speed squared per unit of temperature.
template <typename V4>
__device__ __forceinline__ double cfl_face_dt(double Sfx, double Sfy, double magSf, const double2& g, const V4& wo,
                                              const V4& wn, double c2T, double CFL) {
    const double deltaR = g.x, fraction = g.y;
    const double uxo = wo.y, uyo = wo.z, To = wo.w, uxn = wn.y, uyn = wn.z, Tn = wn.w;
    return CFL * deltaR * magSf /
           ((1.0 - fraction) * fabs(uxo * Sfx + uyo * Sfy) + fraction * fabs(uxn * Sfx + uyn * Sfy) +
            sqrt(c2T * ((1.0 - fraction) * To + fraction * Tn)) * magSf);
}

// Each block reduces a contiguous chunk of faces (stride loop) to one
// partial minimum; the last block to finish reduces the partials and stores
// the time step on the device and, for the host that waits for it, in pinned
// host memory.  Blocks draw tickets by group of kCflGroup, the last of each
// group one more: 1024 tickets on one address, each behind a fence that writes
// the L2 back, took 20 us (250k quads 31 us a launch, so 11.5).  The centres'
// distance and the owner's share of it are stored with the face (16 B) instead
// of formed from its offsets (40 B, a root and a division): 11.5 -> 9.0 us,
// 1.5M triangles 43 -> 30, 740k 24 -> 18.
template <typename R>
__global__ __launch_bounds__(256) void k_cfl(DevPtrs<R> p, double c2T, double CFL, int chunk, double* host_dt) {
    const int blk = xcd_tile(p.map);
    const int f0 = blk * chunk;
    const int f1 = blk < 0 ? f0 : min(p.nf, f0 + chunk);
    double dtf = 1e5;
    for (int f = f0 + threadIdx.x; f < f1; f += 256) {
        const int2 oc = p.fcell[f];
        const double2 sf = p.fsf[f];
        const double d = cfl_face_dt(sf.x, sf.y, p.fmag[f], p.fcfl[f], p.W[oc.x], p.W[oc.y], c2T, CFL);
        dtf = d < dtf ? d : dtf;  // a NaN face value never replaces the minimum
    }
    __shared__ double wmin[4];
    __shared__ int last;
    const double m = block_min_256(dtf, wmin);
    if (threadIdx.x == 0) {
        __hip_atomic_store(&p.dt_part[blockIdx.x], m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned g = blockIdx.x / kCflGroup, ngroups = (gridDim.x + kCflGroup - 1) / kCflGroup;
        const unsigned size = min((unsigned)kCflGroup, gridDim.x - g * kCflGroup);
        // counters one 128-byte line apart: the groups', then the launch's
        unsigned* mine = p.dt_count + 32 * g;
        unsigned* all = p.dt_count + 32 * kCflGroups;
        last = 0;
        // The partial is stored past the L2 (agent scope) and is waited for,
        // and read past it below: no fence, which would write the L2 back.
        // This holds for gfx950, where an agent-scope store that vmcnt has
        // counted is visible to every XCD; the language's memory model would
        // ask for release and acquire here.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (__hip_atomic_fetch_add(mine, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == size - 1) {
            __hip_atomic_store(mine, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (ngroups == 1) {
                last = 1;
            } else if (__hip_atomic_fetch_add(all, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == ngroups - 1) {
                __hip_atomic_store(all, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                last = 1;
            }
        }
    }
    __syncthreads();
    if (!last) return;
    double v = 1e5;
    for (int i = threadIdx.x; i < (int)gridDim.x; i += 256) {
        const double o = __hip_atomic_load(&p.dt_part[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        v = o < v ? o : v;
    }
    v = block_min_256(v, wmin);
    if (threadIdx.x == 0) {
        *p.dt = v;
        if (host_dt) __hip_atomic_store(host_dt, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---------------------------------------------------------------- K5 reconstruct

// 16-byte words of the tile's block of stencil ids (one row of stenW ids per cell).
__device__ __forceinline__ int sten_words(int tile, int tileCells, int nc, int stenW) {
    const int wpt = tileCells >> 6;  // waves per tile
    return min(wpt, ((nc + 63) >> 6) - tile * wpt) * 8 * stenW;
}

// The tile's halo members into LDS slots TILE..: fn(slot, id).
template <int TILE, typename R, typename F>
__device__ __forceinline__ void stage_halo(const DevPtrs<R>& p, int tile, int t, int nthreads, F fn) {
    for (int i = t; i < p.hfix; i += nthreads) fn(TILE + i, p.halo[(size_t)tile * p.hfix + i]);
    const int m0 = p.more_ptr[tile], m1 = p.more_ptr[tile + 1];
    for (int i = m0 + t; i < m1; i += nthreads) fn(TILE + p.hfix + i - m0, p.halo_more[i]);
}

// The reconstructed state of face side i (= 2f + side): FP64 one array per
// variable, FP32 a record plus the temperature again (the layouts of DevPtrs).
template <typename R>
__device__ __forceinline__ void store_face_state(const DevPtrs<R>& p, int i, const typename VT<R>::v4& o) {
    if constexpr (sizeof(R) == 8) {
        p.fvp[i] = o.x;
        p.fvu[i] = o.y;
        p.fvv[i] = o.z;
    } else {
        p.fv[i] = o;
    }
    p.fvT[i] = o.w;
}

// A 16-byte group of coefficients.  Rows of single members (4 or 8 bytes a lane
// and load, up to 17 loads) kept the reconstruction waiting on the loads
// themselves: 740k mixed 79.3 -> 74.6 us with groups, 1.5M FP64 189 -> 184.5,
// 20k quads 8.4 -> 7.7, 17k 8.3 -> 7.5.
template <typename R> struct CoefGroup;
template <> struct CoefGroup<double> {
    using type = double2;
    static __device__ __forceinline__ type splat(double x) { return type{x, x}; }
    static __device__ __forceinline__ double get(const type& g, int i) { return i ? g.y : g.x; }
};
template <> struct CoefGroup<float> {
    using type = float4;
    static __device__ __forceinline__ type splat(float x) { return type{x, x, x, x}; }
    static __device__ __forceinline__ float get(const type& g, int i) {
        return i == 0 ? g.x : i == 1 ? g.y : i == 2 ? g.z : g.w;
    }
};

template <typename R>
__device__ __forceinline__ void limiter_process(R& lim, R& phif, R phic, R phiMax, R phiMin, R gx, R gy, R dx, R dy) {
    // cudaLimiter.h:35-50
    phif = phic + (gx * dx + gy * dy);
    const R d2 = phif - phic;
    const R d1 = (R)(phif < phic) * (phiMin - phic) + (R)(phif >= phic) * (phiMax - phic);
    R yy = fmin((R)2, ((R)0.5 * d1) / ((d2 + (R)(d2 >= (R)0) * K<R>::VSMALL) - (R)(d2 < (R)0) * K<R>::VSMALL));
    const int valid = fabs(d2) >= K<R>::SMALL;
    yy = (R)valid * yy + (R)(1 - valid) * (R)1;
    lim = fmin(lim, yy);
}

// Limiter transforms of K6 (cudaLimiter.h:9-32).
template <typename R> __device__ __forceinline__ R to_bj(R y) { return fmin((R)2 * y, (R)1); }
template <typename R> __device__ __forceinline__ R to_venkat(R y) {
    return fmin((y * y + y + K<R>::VSMALL) / (y * y + (R)0.5 + (R)0.5 * y + K<R>::VSMALL), (R)1);
}

// Whether a flat cell's face states, limiters and BVD temperatures are formed
// where they are read (FP64 at the face centre): the reconstruction then writes
// 40 B per face side and 32 B per cell less, and the face pass reads 64 B per
// face and 32 B per cell less, where the gas is uniform, as ahead of every
// wave.  States and limiters, 1.5M cells, 60% of them on the full path:
// reconstruct 219 -> 192 us, flux 118 -> 114, step 1265 -> 1172; nine corner
// flows 525 -> 480; 20k quads 83.6 -> 83.0; with no flat cell 67.9 -> 68.2.  The
// temperatures too: reconstruct 187 -> 177 us, BVD 18.2 -> 19.2 (it reads the
// flags), step 1136 -> 1117, nine corner flows 456 -> 445, 250k quads 186 ->
// 182; 20k quads and no flat cell 0.3 us longer.  FP32-mixed has half the bytes
// to save and was slower for it (740k cells 469 -> 480).
template <typename R, bool GP> struct FormsFlat {
    static constexpr bool value = sizeof(R) == 8 && !GP;
};

// GP: the flux-quadrature extension's point states (a separate instantiation,
// so the reference path carries none of its registers)
template <typename R, int TILE, bool GP>
__global__ __launch_bounds__(TILE) void k_reconstruct(DevPtrs<R> p) {
    using v4 = typename VT<R>::v4;
    using v2 = typename VT<R>::v2;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    v4* sW = reinterpret_cast<v4*>(smem_raw);
    const int tile = xcd_tile(p.map);
    if (tile < 0) return;
    const int tid = threadIdx.x, c = tile * TILE + tid;
    uint16_t* sRows = reinterpret_cast<uint16_t*>(smem_raw + p.lds_sten_off);
    if (c < p.nc) sW[tid] = p.W[c];
    if (tid == 0) sW[TILE + p.hcap] = v4{(R)1, (R)1, (R)1, (R)1};  // the dummy member
    stage_halo<TILE>(p, tile, tid, TILE, [&](int j, int id) { sW[j] = p.W[id]; });
    {
        const uint4* src = reinterpret_cast<const uint4*>(p.sten + (size_t)tile * TILE * p.stenW);
        const int n16 = sten_words(tile, TILE, p.nc, p.stenW);
        for (int i = tid; i < n16; i += TILE) reinterpret_cast<uint4*>(sRows)[i] = src[i];
    }
    __syncthreads();
    if (c >= p.nc) return;
    const uint16_t* sSt = sRows + tid * p.stenW;  // this cell's members
    const int S = p.scnt[c], C = p.ccnt[c];
    const int maxC = p.maxC;
    const v4 wc = sW[tid];

    R gpx = 0, gpy = 0, guxx = 0, guyx = 0, guxy = 0, guyy = 0, gTx = 0, gTy = 0;
    for (int i = 0; i < C; ++i) {
        const v2 M = p.lsq[sell(c, i, maxC)];
        const v4 wj = sW[sSt[i]];
        R dphi = wj.x - wc.x;
        gpx += M.x * dphi;
        gpy += M.y * dphi;
        dphi = wj.y - wc.y;
        guxx += M.x * dphi;
        guyx += M.y * dphi;
        dphi = wj.z - wc.z;
        guxy += M.x * dphi;
        guyy += M.y * dphi;
        dphi = wj.w - wc.w;
        gTx += M.x * dphi;
        gTy += M.y * dphi;
    }
    p.gp[c] = v2{gpx, gpy};
    p.gu[c] = v2{guxx, guyx};
    p.gv[c] = v2{guxy, guyy};
    p.gT[c] = v2{gTx, gTy};

    R pMax = wc.x, pMin = wc.x, uxMax = wc.y, uxMin = wc.y, uyMax = wc.z, uyMin = wc.z, TMax = wc.w, TMin = wc.w;
    for (int i = 0; i < C; ++i) {
        const v4 wj = sW[sSt[i]];
        pMax = fmax(wj.x, pMax);
        pMin = fmin(wj.x, pMin);
        uxMax = fmax(wj.y, uxMax);
        uxMin = fmin(wj.y, uxMin);
        uyMax = fmax(wj.z, uyMax);
        uyMin = fmin(wj.z, uyMin);
        TMax = fmax(wj.w, TMax);
        TMin = fmin(wj.w, TMin);
    }

    const int nf = p.nf;
    // as in k_reconstruct_q: the cells whose face states and limiters the face pass forms
    const bool flat = fabs(TMax - TMin) < K<R>::VSMALL;
    bool skip = false;
    if constexpr (FormsFlat<R, GP>::value) {
        bool edge = false;
        if (p.boundaryFirstOrder)
            for (int fi = 0; fi < C; ++fi) edge = edge || abs(p.slot_face[sell(c, fi, maxC)]) - 1 >= nf;
        skip = flat && !edge;
        const bool wasFlat = p.flat_prev[c] != 0;
        if (flat != wasFlat) {
            p.flat_prev[c] = flat;
            for (int fi = 0; fi < C; ++fi) {
                const int sf = p.slot_face[sell(c, fi, maxC)];
                const int f = (sf < 0 ? -sf : sf) - 1;
                if (f < nf) p.fflat[2 * f + (sf < 0)] = skip;
            }
        }
    }
    if (flat) {
        const bool store = !skip || p.storeFlat;
        if (store) p.lim[c] = v4{(R)1, (R)1, (R)1, (R)1};
        const R lT = to_bj((R)1);  // the BVD test's limiter of this cell
        p.tlim[c] = lT < K<R>::VALID_LIM_FACTOR;
        for (int fi = 0; fi < C; ++fi) {
            const int sf = p.slot_face[sell(c, fi, maxC)];
            const int isNei = sf < 0;
            const int f = (sf < 0 ? -sf : sf) - 1;
            if (f >= nf) continue;
            const v2 d = p.slot_d[sell(c, fi, maxC)];
            const R dx = d.x, dy = d.y;
            if (!store) continue;
            v4 o;
            o.x = wc.x + gpx * dx + gpy * dy;
            o.y = wc.y + guxx * dx + guyx * dy;
            o.z = wc.z + guxy * dx + guyy * dy;
            o.w = wc.w + gTx * dx + gTy * dy;
            store_face_state(p, 2 * f + isNei, o);
            p.tTVD[sell(c, fi, maxC)] = wc.w + lT * (gTx * dx + gTy * dy);
            if constexpr (GP)
                for (int g = 0; g < p.ngp; ++g) {  // flux points (extension): the same linear state there
                const v4 dg = p.fgd[(size_t)g * nf + f];
                const R gx = (R)(isNei ? dg.z : dg.x), gy = (R)(isNei ? dg.w : dg.y);
                v4 og;
                og.x = wc.x + gpx * gx + gpy * gy;
                og.y = wc.y + guxx * gx + guyx * gy;
                og.z = wc.z + guxy * gx + guyy * gy;
                og.w = wc.w + gTx * gx + gTy * gy;
                p.fvg[((size_t)g * nf + f) * 2 + isNei] = og;
            }
        }
        p.smooth[c] = 0;
        return;
    }

    // RBF sum over row k of K per slice (DevLayout::rbf_at): eight members at a
    // time, their ids one 16-byte word, their coefficients 16-byte groups requested
    // together; the last group's members past the stencil add -0.0 * 1.  Bound by
    // its loads: one id and one coefficient a load, which read half or a quarter of
    // each group, took 123.4 us on 735k triangles and quads in FP32-mixed (so
    // 106.5; FP64 64.9, 60.0), 23.0 on 180k periodic triangles (21.5; FP64 35.0,
    // 34.1), at two flux points on 135k 67.1 (48; FP64 73.8, 55.7).
    constexpr int V = 16 / sizeof(R);
    using G = typename CoefGroup<R>::type;
    const uint4* row = reinterpret_cast<const uint4*>(sSt);
    auto rbf_sum = [&](const R* rbf, int k, int K) {
        const R* a = rbf + ((size_t)(c >> 6) * K + k) * p.rbfRow;
        const G* groups = reinterpret_cast<const G*>(a + 64) + (c & 63);
        const R own = a[c & 63];
        v4 o = {own * wc.x, own * wc.y, own * wc.z, own * wc.w};
        for (int j0 = 0; j0 < S; j0 += 8) {
            const uint4 ids = row[j0 >> 3];
            const unsigned w[4] = {ids.x, ids.y, ids.z, ids.w};
            G gs[8 / V];
#pragma unroll
            for (int j = 0; j < 8; j += V)
                if (j0 + j < S) gs[j / V] = groups[(j0 + j) / V * 64];
#pragma unroll
            for (int j = 0; j < 8; j += V) {
                if (j0 + j >= S) break;
                const G g = gs[j / V];
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int h = j + i;
                    const v4 m = sW[(h & 1) ? w[h >> 1] >> 16 : w[h >> 1] & 0xffffu];
                    const R coef = CoefGroup<R>::get(g, i);
                    o.x += coef * m.x;
                    o.y += coef * m.y;
                    o.z += coef * m.z;
                    o.w += coef * m.w;
                }
            }
        }
        return o;
    };

    R limP = 2, limUx = 2, limUy = 2, limT = 2;
    R smoothness = 0;
    int isNotTrouble = 1;
    const R rP = fabs(pMax - pMin), rUx = fabs(uxMax - uxMin), rUy = fabs(uyMax - uyMin), rT = fabs(TMax - TMin);
    for (int fi = 0; fi < C; ++fi) {
        const int sf = p.slot_face[sell(c, fi, maxC)];
        const int isNei = sf < 0;
        const int f = (sf < 0 ? -sf : sf) - 1;
        if (f >= nf) continue;
        const v2 d = p.slot_d[sell(c, fi, maxC)];
        const R dx = d.x, dy = d.y;
        const R deltaR = p.slot_dr[sell(c, fi, maxC)];
        const R fraction = sqrt(dx * dx + dy * dy) / deltaR;
        const int nbl = sSt[fi];

        const v4 of = rbf_sum(p.rbf, fi, maxC);
        const R pf = of.x, uxf = of.y, uyf = of.z, Tf = of.w;
        v4 o;
        R phif;
        limiter_process(limP, phif, wc.x, pMax, pMin, gpx, gpy, dx, dy);
        o.x = (R)(rP >= K<R>::SMALL) * pf + (R)(rP < K<R>::SMALL) * phif;
        isNotTrouble = phif > (R)0;
        smoothness = fmax(smoothness, fabs(((R)1 - fraction) * wc.x + fraction * sW[nbl].x - phif) / deltaR +
                                          (R)(pf <= (R)0) * (R)1e20 + (R)(phif <= (R)0) * (R)1e20);
        limiter_process(limUx, phif, wc.y, uxMax, uxMin, guxx, guyx, dx, dy);
        o.y = (R)(rUx >= K<R>::SMALL) * uxf + (R)(rUx < K<R>::SMALL) * phif;
        limiter_process(limUy, phif, wc.z, uyMax, uyMin, guxy, guyy, dx, dy);
        o.z = (R)(rUy >= K<R>::SMALL) * uyf + (R)(rUy < K<R>::SMALL) * phif;
        limiter_process(limT, phif, wc.w, TMax, TMin, gTx, gTy, dx, dy);
        o.w = (R)(rT >= K<R>::SMALL) * Tf + (R)(rT < K<R>::SMALL) * phif;
        isNotTrouble = phif > (R)0;
        store_face_state(p, 2 * f + isNei, o);
        if constexpr (GP)
        for (int g = 0; g < p.ngp; ++g) {  // flux points (extension), as in k_reconstruct_q
            const v4 q = rbf_sum(p.rbf_gp, g * maxC + fi, p.ngp * maxC);
            const R pg = q.x, uxg = q.y, uyg = q.z, Tg = q.w;
            const v4 dg = p.fgd[(size_t)g * nf + f];
            const R gx = (R)(isNei ? dg.z : dg.x), gy = (R)(isNei ? dg.w : dg.y);
            v4 og;
            og.x = (R)(rP >= K<R>::SMALL) * pg + (R)(rP < K<R>::SMALL) * (wc.x + (gpx * gx + gpy * gy));
            og.y = (R)(rUx >= K<R>::SMALL) * uxg + (R)(rUx < K<R>::SMALL) * (wc.y + (guxx * gx + guyx * gy));
            og.z = (R)(rUy >= K<R>::SMALL) * uyg + (R)(rUy < K<R>::SMALL) * (wc.z + (guxy * gx + guyy * gy));
            og.w = (R)(rT >= K<R>::SMALL) * Tg + (R)(rT < K<R>::SMALL) * (wc.w + (gTx * gx + gTy * gy));
            p.fvg[((size_t)g * nf + f) * 2 + isNei] = og;
        }
    }
    const R nt = (R)isNotTrouble;
    const R limTraw = fmax(limT, (R)0) * nt;
    p.lim[c] = v4{fmax(limP, (R)0) * nt, fmax(limUx, (R)0) * nt, fmax(limUy, (R)0) * nt, limTraw};
    smoothness = smoothness / ((R)0.5 * (pMax + pMin) * nt + K<R>::VSMALL);
    p.smooth[c] = smoothness > (R)1;
    // the BVD test's inputs of this cell (cudaLimiter.h:431-440): its limiter
    // condition and the limited linear temperature on each internal face
    const R lT = to_bj(limTraw);
    p.tlim[c] = lT < K<R>::VALID_LIM_FACTOR;
    for (int fi = 0; fi < C; ++fi) {
        const int sf = p.slot_face[sell(c, fi, maxC)];
        const int f = (sf < 0 ? -sf : sf) - 1;
        if (f >= nf) continue;
        const v2 d = p.slot_d[sell(c, fi, maxC)];
        p.tTVD[sell(c, fi, maxC)] = wc.w + lT * (gTx * d.x + gTy * d.y);
    }
}

// Moves within groups of four consecutive lanes (DPP quad permutations, full
// rate VALU); every lane of the group must be active.
template <int CTRL> __device__ __forceinline__ int dpp_move(int x) {
    return __builtin_amdgcn_mov_dpp(x, CTRL, 0xF, 0xF, false);
}
template <int CTRL> __device__ __forceinline__ float dpp_move(float x) {
    return __int_as_float(dpp_move<CTRL>(__float_as_int(x)));
}
template <int CTRL> __device__ __forceinline__ double dpp_move(double x) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = (unsigned)dpp_move<CTRL>((int)(unsigned)u);
    const unsigned hi = (unsigned)dpp_move<CTRL>((int)(unsigned)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// the value of lane J of this lane's group
template <int J, typename T> __device__ __forceinline__ T quad_bcast(T x) { return dpp_move<J * 0x55>(x); }
// the value of lane (this lane xor X) of the group, X = 1 or 2
template <int X, typename T> __device__ __forceinline__ T quad_xor(T x) {
    return dpp_move<X == 1 ? 0xB1 : 0x4E>(x);  // quad_perm [1,0,3,2] and [2,3,0,1]
}

// The largest of the values below 32 that x has in the lanes where m holds (0
// if there is none): the same in every lane.
__device__ __forceinline__ int wave_max32(int x, bool m) {
    int r = 0;
#pragma unroll
    for (int b = 16; b > 0; b >>= 1)
        if (__ballot(m && x >= r + b) != 0) r += b;
    return r;
}

// K5 with four lanes per cell, for meshes whose cells have at most four
// faces (triangles and quads): lane k of a cell's group handles face slot k
// (its RBF sum and limiter candidates) and variable k of the gradient and the
// compact min/max, which the group then shares.  The per-cell results are
// exact reductions over the group (the limiter is a minimum, the smoothness a
// maximum, the trouble test that of the last internal face), so the values
// equal the one-lane-per-cell kernel's bit for bit.
// MS bounds the stencil size (8: quads, 16: mixed triangles and quads, 20), so
// that meshes of short stencils hold fewer coefficients in registers.
//
// Bound by its chain of loads and LDS reads on small meshes (15.8k cycles per
// wave before the following), by the memory it writes and by VALU issue on
// large ones.  No step of the chain waits alone: halo ids lie in rows of fixed
// width (no offset to wait for), slots are read without their count, a cell's
// member ids are one or two 16-byte words, and the RBF sums run to the
// wavefront's longest stencil with terms that add nothing past a cell's own.
// Back to back: 800 cells 8.3 -> 6.2 us, 20k quads 10.1 -> 8.4 (mixed 7.9 ->
// 6.5), 17k periodic quads 9.7 -> 8.3, 524k mixed 44.1 -> 41.1; 1.5M triangles
// and quads 221 -> 220.
// Waves per SIMD the register allocator must allow, per working type
// (build-time tuning knobs; 1 = no constraint).  At 5 (FP64) and 8 (FP32) the
// 16-member kernels spill 5 values and 1: Riemann 233 us instead of 220, and
// 84.4 instead of 81.2 (mixed, 740k cells).
#ifndef AFAR_RECONQ_WPE_D
#define AFAR_RECONQ_WPE_D 4
#endif
#ifndef AFAR_RECONQ_WPE_F
#define AFAR_RECONQ_WPE_F 7
#endif
// The instantiations for flux points and (float) for stencils of 20 hold more
// values and ask for fewer waves, so that none spills.  With flux points, float
// stencils past 8 at 5 waves spilled 4 to 8 values: 240k triangles and quads
// 61.0 us, at 4 waves 54.7.
template <typename R, bool GP, int MS> struct ReconQWaves {
    static constexpr int value = sizeof(R) == 8 ? AFAR_RECONQ_WPE_D - (GP ? 1 : 0)
                                                : AFAR_RECONQ_WPE_F - (GP ? (MS > 8 ? 3 : 2) : MS > 16 ? 1 : 0);
};
#define AFAR_RECONQ_ATTR __attribute__((amdgpu_waves_per_eu(ReconQWaves<R, GP, MS>::value, 8)))

template <typename R, int TILE, bool GP, int MS>
__global__ __launch_bounds__(4 * TILE) AFAR_RECONQ_ATTR void k_reconstruct_q(DevPtrs<R> p) {
    using v4 = typename VT<R>::v4;
    using v2 = typename VT<R>::v2;
    constexpr int NT = 4 * TILE;
    // FP64 at the face centre: lane k forms its slot's geometry (face offset,
    // neighbour offset and distance) and least-squares weight from the staged
    // cell centres and the face centre, with k_lsq's and the host layout's
    // operations in their order, instead of reading 40 bytes of stored slot
    // data per slot; the weights are shared within the group by DPP.
    constexpr bool GEO = sizeof(R) == 8 && !GP;
    constexpr bool FLAT = FormsFlat<R, GP>::value;
    // Flux points: a point's coefficients are requested at once, before its sum,
    // where the registers for them are there.  A block of 1024 threads leaves a
    // thread 128, which FP64 stencils past 8 need for the rest: requested at once
    // they spill 25 values and more, 240k triangles and quads in tiles of 256
    // 83.8 us, group by group 72.6.
    constexpr bool AHEAD = !(sizeof(R) == 8 && TILE == 256 && MS > 8);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    v4* sW = reinterpret_cast<v4*>(smem_raw);
    uint16_t* sRows = reinterpret_cast<uint16_t*>(smem_raw + p.lds_sten_off);
    v2* sM = reinterpret_cast<v2*>(smem_raw + p.lds_m_off);            // 4 weights per cell
    double2* sC = reinterpret_cast<double2*>(smem_raw + p.lds_m_off);  // GEO: tile + halo centres instead
    const int tile = xcd_tile(p.map);
    if (tile < 0) return;
    const int t = threadIdx.x;
    const int lc = t >> 2, k = t & 3;
    const int c0 = tile * TILE, c = c0 + lc;
    const int maxC = p.maxC, nf = p.nf, SW = p.stenW;
    // Cell and slot arrays are addressed from bases the wavefront shares (its
    // 16 cells lie in one slice) with small lane offsets: scalar address
    // arithmetic instead of 64-bit vector arithmetic (with tTVD stored in slot
    // order: 740k mixed 81.4 -> 79.3 us, BVD 9.9 -> 9.2; 1.5M FP64 222 -> 220).
    const size_t slice = (unsigned)(c0 + 16 * __builtin_amdgcn_readfirstlane(t >> 6)) >> 6;
    const unsigned cl = c & 63, row_k = k * 64 + cl;
    auto slots = [&](auto* a) { return a + slice * maxC * 64; };  // [row_k]: lane k's slot
    // Every load that needs no LDS is issued before the staging barrier, in
    // two dependent rounds: (1) the cell's counts, lane k's slot, the tile's
    // own states, halo ids and stencil rows; (2) the halo states, the slot's
    // face centre and, where the full path is foreseen, its RBF coefficients.
    const bool inb = c < p.nc;
    int S = 0, C = 0, sf = 0, wasFlat = 0;
    if (inb) {
        S = (p.scnt + c0)[lc];
        C = (p.ccnt + c0)[lc];
        wasFlat = (p.flat_prev + c0)[lc];
        if (k < maxC) sf = slots(p.slot_face)[row_k];  // 0: no such slot
    }
    const int n16 = sten_words(tile, TILE, p.nc, SW);
    const uint4* stSrc = reinterpret_cast<const uint4*>(p.sten + (size_t)tile * TILE * SW);
    const bool ownW = t < TILE && tile * TILE + t < p.nc;
    const bool ownH = t < p.hfix;
    v4 wOwn, wHalo;
    double2 cOwn, cHalo;  // GEO: staged centres
    uint4 st0;
    int h0 = 0;
    if (ownH) h0 = (p.halo + (size_t)tile * p.hfix)[t];
    if (ownW) {
        wOwn = (p.W + c0)[t];
        if constexpr (GEO) cOwn = (p.cen + c0)[t];
    }
    if (t < n16) st0 = stSrc[t];
    const int m0 = p.more_ptr[tile], m1 = p.more_ptr[tile + 1];
    if (ownH) {
        wHalo = p.W[h0];
        if constexpr (GEO) cHalo = p.cen[h0];
    }
    const int isNei = sf < 0;
    const int f = (sf < 0 ? -sf : sf) - 1;
    const bool has = sf != 0, live = has && f < nf;
    v2 Mk = v2{(R)0, (R)0};
    v2 d = v2{(R)0, (R)0};
    double2 fc = double2{0.0, 0.0}, fs = double2{0.0, 0.0};  // GEO: face centre, periodic shift
    if (has) {
        if constexpr (GEO) {
            fc = p.fcen[f];
            if (p.fshift && live) fs = p.fshift[f];
        } else {
            Mk = slots(p.lsq)[row_k];
            d = slots(p.slot_d)[row_k];
        }
    }
    // A cell that took the full path at the previous launch most likely takes
    // it again: its RBF coefficients and centre distance are requested in this
    // round already.  (flat_prev is more than this hint: the writes of fflat
    // below, which say whose states the face pass forms, are left out where it
    // says that nothing changed, so both arrays are written by this kernel alone
    // and together.)  The row count is the wavefront's: a cell of a shorter stencil reads
    // its padding (-0.0), which shares the other cells' 128-byte segments.
    constexpr int V = 16 / sizeof(R), NG = (MS + V - 1) / V;  // members per 16-byte group, groups
    using G = typename CoefGroup<R>::type;
    R cf0 = (R)-0.0;  // the cell's own coefficient
    G cf[NG];         // the members'
    R deltaR = 0;
    const R* a = p.rbf + slice * maxC * p.rbfRow;  // this slice's rows; lane k's at k * rbfRow
    const unsigned a0 = k * p.rbfRow + cl, a1 = (k * p.rbfRow + 64) / V + cl;
#pragma unroll
    for (int i = 0; i < NG; ++i) cf[i] = CoefGroup<R>::splat((R)-0.0);
    auto load_coefficients = [&](bool need) {
        const int rows = wave_max32(S, need);
        if (need) {
            if constexpr (!GEO) deltaR = slots(p.slot_dr)[row_k];
            cf0 = a[a0];
#pragma unroll
            for (int i = 0; i < NG; ++i)
                if (i * V < rows) cf[i] = (reinterpret_cast<const G*>(a) + i * 64)[a1];
        }
    };
    const bool early = live && !wasFlat;
    load_coefficients(early);
    uint4* stDst = reinterpret_cast<uint4*>(sRows);
    if (ownW) {
        sW[t] = wOwn;
        if constexpr (GEO) sC[t] = cOwn;
    }
    if (ownH) {
        sW[TILE + t] = wHalo;
        if constexpr (GEO) sC[TILE + t] = cHalo;
    }
    if (t < n16) stDst[t] = st0;
    if constexpr (!GEO) sM[t] = Mk;
    if (t == NT - 1) sW[TILE + p.hcap] = v4{(R)1, (R)1, (R)1, (R)1};  // the dummy member
    auto stage = [&](int j, int id) {
        sW[j] = p.W[id];
        if constexpr (GEO) sC[j] = p.cen[id];
    };
    for (int i = t + NT; i < p.hfix; i += NT) stage(TILE + i, p.halo[(size_t)tile * p.hfix + i]);
    for (int i = m0 + t; i < m1; i += NT) stage(TILE + p.hfix + i - m0, p.halo_more[i]);
    for (int i = t + NT; i < n16; i += NT) stDst[i] = stSrc[i];
    __syncthreads();
    if (!inb) return;  // the four lanes of a cell leave together
    const R* sWr = reinterpret_cast<const R*>(sW);

    // the cell's member ids, eight to a 16-byte word; its compact neighbours
    // (the cell itself where it has fewer than four)
    const uint4* row = reinterpret_cast<const uint4*>(sRows + lc * SW);
    const uint4 row0 = row[0];
    const int nb[4] = {C > 0 ? (int)(row0.x & 0xffffu) : lc, C > 1 ? (int)(row0.x >> 16) : lc,
                       C > 2 ? (int)(row0.y & 0xffffu) : lc, C > 3 ? (int)(row0.y >> 16) : lc};
    const int nbl = (k & 2) ? ((k & 1) ? nb[3] : nb[2]) : ((k & 1) ? nb[1] : nb[0]);  // across lane k's slot

    // the temperature range over the compact stencil selects the branch
    R TMax = sWr[4 * lc + 3], TMin = TMax;
    {
        R Tj[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) Tj[i] = sWr[4 * nb[i] + 3];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            TMax = fmax(Tj[i], TMax);
            TMin = fmin(Tj[i], TMin);
        }
    }
    double ex = 0.0, ey = 0.0;  // GEO: compact neighbour - cell centre of lane k's slot
    if constexpr (GEO) {
        // the host layout's expressions (face offset d, neighbour offset e):
        // from the neighbour side the cell is seen shifted, from the owner's
        // the neighbour; no shift enters at a boundary face
        const double2 cc = sC[lc], cn = sC[nbl];
        const double ax = live && isNei ? cc.x + fs.x : cc.x, ay = live && isNei ? cc.y + fs.y : cc.y;
        const double bx = live && !isNei ? cn.x + fs.x : cn.x, by = live && !isNei ? cn.y + fs.y : cn.y;
        if (has) {
            d = v2{fc.x - ax, fc.y - ay};
            ex = bx - ax;
            ey = by - ay;
        }
        // k_lsq's sums over the compact slots in order, then lane k's weight;
        // a lane without a slot adds 0 * 0
        double Sxx = 0.0, Sxy = 0.0, Syy = 0.0;
        const double qx[4] = {quad_bcast<0>(ex), quad_bcast<1>(ex), quad_bcast<2>(ex), quad_bcast<3>(ex)};
        const double qy[4] = {quad_bcast<0>(ey), quad_bcast<1>(ey), quad_bcast<2>(ey), quad_bcast<3>(ey)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            Sxx += qx[i] * qx[i];
            Sxy += qx[i] * qy[i];
            Syy += qy[i] * qy[i];
        }
        const double det = Sxx * Syy - Sxy * Sxy;
        const v2 m = v2{(Syy * ex - Sxy * ey) / det, (-Sxy * ex + Sxx * ey) / det};
        if (has) Mk = m;
    }
    // Lane k forms variable k's least-squares gradient and compact-stencil
    // extrema (the reference's per-variable sums, in the same order; the
    // extrema are exact) and stores the gradient; the group then shares them.
    // The full path does this after its RBF sums, so that fewer values are
    // live while the coefficients are in registers.  A missing neighbour adds
    // 0 * 0, which leaves the sums (never -0) as they are.
    R gxk = 0, gyk = 0, mxk = 0, mnk = 0;
    auto gradient = [&]() {
        const R wck = sWr[4 * lc + k];
        mxk = wck;
        mnk = wck;
        R cj[4];
        v2 M[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            cj[i] = sWr[4 * nb[i] + k];
            if constexpr (!GEO) M[i] = sM[4 * lc + i];
        }
        if constexpr (GEO) {  // every slot's weight from its lane
            M[0] = v2{quad_bcast<0>(Mk.x), quad_bcast<0>(Mk.y)};
            M[1] = v2{quad_bcast<1>(Mk.x), quad_bcast<1>(Mk.y)};
            M[2] = v2{quad_bcast<2>(Mk.x), quad_bcast<2>(Mk.y)};
            M[3] = v2{quad_bcast<3>(Mk.x), quad_bcast<3>(Mk.y)};
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const R dphi = i < C ? cj[i] - wck : (R)0;
            gxk += M[i].x * dphi;
            gyk += M[i].y * dphi;
            mxk = fmax(cj[i], mxk);
            mnk = fmin(cj[i], mnk);
        }
        v2* g = k == 0 ? p.gp : k == 1 ? p.gu : k == 2 ? p.gv : p.gT;
        (g + c0)[lc] = v2{gxk, gyk};
    };
    const bool flat = fabs(TMax - TMin) < K<R>::VSMALL;

    if (k == 0 && flat != (wasFlat != 0)) (p.flat_prev + c0)[lc] = flat;
    // The face pass forms a flat cell's face states and limiters itself
    // (DevPtrs::fflat); a first-order boundary cell's limiter is the BVD pass's.
    bool edge = false;
    if (FLAT && p.boundaryFirstOrder) edge = ((__ballot(has && !live) >> ((t & 63) & ~3)) & 0xF) != 0;
    const bool skip = FLAT && flat && !edge;
    if (FLAT && live && skip != (wasFlat && !edge)) p.fflat[2 * f + isNei] = skip;
    // Full path not foreseen: every RBF coefficient of the face and its centre
    // distance are requested now, at once (one memory round trip).
    const bool late = !flat && live && !early;
    if (__any(late)) load_coefficients(late);
    if constexpr (GEO) {
        if (!flat && live) deltaR = afar_hypot(ex, ey);  // k_lsq's centre distance
    }
    const R dx = d.x, dy = d.y;
    const v4 wc = sW[lc];
    if (flat) {
        gradient();
        const R gpx = quad_bcast<0>(gxk), gpy = quad_bcast<0>(gyk), guxx = quad_bcast<1>(gxk),
                guyx = quad_bcast<1>(gyk), guxy = quad_bcast<2>(gxk), guyy = quad_bcast<2>(gyk),
                gTx = quad_bcast<3>(gxk), gTy = quad_bcast<3>(gyk);
        const R lT = to_bj((R)1);  // the BVD test's limiter of this cell
        const bool store = !skip || p.storeFlat;
        if (k == 0) {
            if (store) (p.lim + c0)[lc] = v4{(R)1, (R)1, (R)1, (R)1};
            (p.smooth + c0)[lc] = 0;
            (p.tlim + c0)[lc] = lT < K<R>::VALID_LIM_FACTOR;
        }
        if (live && store) {
            v4 o;
            o.x = wc.x + gpx * dx + gpy * dy;
            o.y = wc.y + guxx * dx + guyx * dy;
            o.z = wc.z + guxy * dx + guyy * dy;
            o.w = wc.w + gTx * dx + gTy * dy;
            store_face_state(p, 2 * f + isNei, o);
            slots(p.tTVD)[row_k] = wc.w + lT * (gTx * dx + gTy * dy);
            if constexpr (GP)
                for (int g = 0; g < p.ngp; ++g) {  // flux points (extension): the same linear state there
                const v4 dg = p.fgd[(size_t)g * nf + f];
                const R gx = (R)(isNei ? dg.z : dg.x), gy = (R)(isNei ? dg.w : dg.y);
                v4 og;
                og.x = wc.x + gpx * gx + gpy * gy;
                og.y = wc.y + guxx * gx + guyx * gy;
                og.z = wc.z + guxy * gx + guyy * gy;
                og.w = wc.w + gTx * gx + gTy * gy;
                p.fvg[((size_t)g * nf + f) * 2 + isNei] = og;
            }
        }
        return;
    }

    // RBF sums, a group of members at a time up to the wavefront's longest
    // stencil: the states of a group are requested together, and a cell that
    // has no further members adds -0.0 * 1.
    const int rows = wave_max32(S, live);
    auto rbf_sum = [&](R own, auto group, v4& o) {
        o = v4{own * wc.x, own * wc.y, own * wc.z, own * wc.w};
        uint4 ids = row0;
#pragma unroll
        for (int j = 0; j < NG * V; j += V) {
            if (j < rows) {
                if (j == 8 || j == 16) ids = row[j / 8];
                const G g = group(j / V);
                const unsigned w[4] = {ids.x, ids.y, ids.z, ids.w};
                v4 m[V];
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int h = (j + i) & 7;
                    m[i] = sW[(h & 1) ? w[h >> 1] >> 16 : w[h >> 1] & 0xffffu];
                }
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const R coef = CoefGroup<R>::get(g, i);
                    o.x += coef * m[i].x;
                    o.y += coef * m[i].y;
                    o.z += coef * m[i].z;
                    o.w += coef * m[i].w;
                }
            }
        }
    };
    v4 of;
    rbf_sum(cf0, [&](int i) { return cf[i]; }, of);
    const R pf = of.x, uxf = of.y, uyf = of.z, Tf = of.w;
    gradient();
    const R gpx = quad_bcast<0>(gxk), gpy = quad_bcast<0>(gyk), guxx = quad_bcast<1>(gxk),
            guyx = quad_bcast<1>(gyk), guxy = quad_bcast<2>(gxk), guyy = quad_bcast<2>(gyk),
            gTx = quad_bcast<3>(gxk), gTy = quad_bcast<3>(gyk);
    const R pMax = quad_bcast<0>(mxk), pMin = quad_bcast<0>(mnk), uxMax = quad_bcast<1>(mxk),
            uxMin = quad_bcast<1>(mnk), uyMax = quad_bcast<2>(mxk), uyMin = quad_bcast<2>(mnk);

    R limP = 2, limUx = 2, limUy = 2, limT = 2;
    R smoothness = 0;
    int faceNotTrouble = 1;
    if (live) {
        const R rP = fabs(pMax - pMin), rUx = fabs(uxMax - uxMin), rUy = fabs(uyMax - uyMin), rT = fabs(TMax - TMin);
        v4 o;
        R phif;
        const R fraction = sqrt(dx * dx + dy * dy) / deltaR;
        limiter_process(limP, phif, wc.x, pMax, pMin, gpx, gpy, dx, dy);
        o.x = (R)(rP >= K<R>::SMALL) * pf + (R)(rP < K<R>::SMALL) * phif;
        smoothness = fmax(smoothness, fabs(((R)1 - fraction) * wc.x + fraction * sW[nbl].x - phif) / deltaR +
                                          (R)(pf <= (R)0) * (R)1e20 + (R)(phif <= (R)0) * (R)1e20);
        limiter_process(limUx, phif, wc.y, uxMax, uxMin, guxx, guyx, dx, dy);
        o.y = (R)(rUx >= K<R>::SMALL) * uxf + (R)(rUx < K<R>::SMALL) * phif;
        limiter_process(limUy, phif, wc.z, uyMax, uyMin, guxy, guyy, dx, dy);
        o.z = (R)(rUy >= K<R>::SMALL) * uyf + (R)(rUy < K<R>::SMALL) * phif;
        limiter_process(limT, phif, wc.w, TMax, TMin, gTx, gTy, dx, dy);
        o.w = (R)(rT >= K<R>::SMALL) * Tf + (R)(rT < K<R>::SMALL) * phif;
        faceNotTrouble = phif > (R)0;
        store_face_state(p, 2 * f + isNei, o);
        // flux points (extension): RBF sums with the point's coefficients,
        // or the unlimited linear state where the compact range is flat
        if constexpr (GP)
        for (int g = 0; g < p.ngp; ++g) {
            const R* ag = p.rbf_gp + (slice * p.ngp + g) * maxC * p.rbfRow;
            auto group = [&](int i) { return (reinterpret_cast<const G*>(ag) + i * 64)[a1]; };
            cf0 = ag[a0];
            v4 q;
            if constexpr (AHEAD) {
#pragma unroll
                for (int i = 0; i < NG; ++i)
                    if (i * V < rows) cf[i] = group(i);
                rbf_sum(cf0, [&](int i) { return cf[i]; }, q);
            } else {
                rbf_sum(cf0, group, q);
            }
            const R pg = q.x, uxg = q.y, uyg = q.z, Tg = q.w;
            const v4 dg = p.fgd[(size_t)g * nf + f];
            const R gx = (R)(isNei ? dg.z : dg.x), gy = (R)(isNei ? dg.w : dg.y);
            v4 og;
            og.x = (R)(rP >= K<R>::SMALL) * pg + (R)(rP < K<R>::SMALL) * (wc.x + (gpx * gx + gpy * gy));
            og.y = (R)(rUx >= K<R>::SMALL) * uxg + (R)(rUx < K<R>::SMALL) * (wc.y + (guxx * gx + guyx * gy));
            og.z = (R)(rUy >= K<R>::SMALL) * uyg + (R)(rUy < K<R>::SMALL) * (wc.z + (guxy * gx + guyy * gy));
            og.w = (R)(rT >= K<R>::SMALL) * Tg + (R)(rT < K<R>::SMALL) * (wc.w + (gTx * gx + gTy * gy));
            p.fvg[((size_t)g * nf + f) * 2 + isNei] = og;
        }
    }
    // group reductions (lanes 4j..4j+3 of the wavefront)
    limP = fmin(limP, quad_xor<1>(limP));
    limUx = fmin(limUx, quad_xor<1>(limUx));
    limUy = fmin(limUy, quad_xor<1>(limUy));
    limT = fmin(limT, quad_xor<1>(limT));
    smoothness = fmax(smoothness, quad_xor<1>(smoothness));
    limP = fmin(limP, quad_xor<2>(limP));
    limUx = fmin(limUx, quad_xor<2>(limUx));
    limUy = fmin(limUy, quad_xor<2>(limUy));
    limT = fmin(limT, quad_xor<2>(limT));
    smoothness = fmax(smoothness, quad_xor<2>(smoothness));
    // the trouble test of the last internal face in slot order
    const unsigned long long lm = __ballot(live);
    const int base = (t & 63) & ~3;
    const unsigned grp = (unsigned)(lm >> base) & 0xFu;
    const int lastLane = grp ? 31 - __builtin_clz(grp) : 0;
    const int nt0 = __shfl(faceNotTrouble, base + lastLane);
    const int isNotTrouble = grp ? nt0 : 1;
    const R nt = (R)isNotTrouble;
    const R limTraw = fmax(limT, (R)0) * nt;
    // the BVD test's inputs (cudaLimiter.h:431-440): the limited linear
    // temperature on lane k's face, and the cell's limiter condition
    const R lT = to_bj(limTraw);
    if (live) slots(p.tTVD)[row_k] = wc.w + lT * (gTx * dx + gTy * dy);
    if (k == 0) {
        (p.lim + c0)[lc] = v4{fmax(limP, (R)0) * nt, fmax(limUx, (R)0) * nt, fmax(limUy, (R)0) * nt, limTraw};
        smoothness = smoothness / ((R)0.5 * (pMax + pMin) * nt + K<R>::VSMALL);
        (p.smooth + c0)[lc] = smoothness > (R)1;
        (p.tlim + c0)[lc] = lT < K<R>::VALID_LIM_FACTOR;
    }
}

// ---------------------------------------------------------------- K6 BVD indicator


template <typename R, int TILE>
__global__ __launch_bounds__(TILE) void k_bvd(DevPtrs<R> p) {
    using v4 = typename VT<R>::v4;
    constexpr int PF = 4;  // face slots whose data is requested in the first load rounds
    constexpr bool FLAT = FormsFlat<R, false>::value;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    int8_t* sS = reinterpret_cast<int8_t*>(smem_raw);
    uint16_t* sSt = reinterpret_cast<uint16_t*>(smem_raw + p.lds_bvd_sten_off);
    const int tile = xcd_tile(p.map);
    if (tile < 0) return;
    const int tid = threadIdx.x, c0 = tile * TILE, c = c0 + tid;
    const int maxC = p.maxC, nf = p.nf;
    const bool inb = c < p.nc;
    // Two rounds of independent loads before the tile's flag vote: (1) the cell's
    // counts, flag and limiter condition, the first slots' faces and halo
    // ids; (2) halo flags and, in cells meeting the limiter condition, the
    // slots' face temperatures (both sides' O3 values and this side's limited
    // linear value, formed by the reconstruction).  Halo and stencil indices
    // are clamped rather than branched on, and values held in plain scalars,
    // so that no load is waited for before its round is complete.  The
    // stencil block is read only by tiles with a flagged cell among their own
    // and halo cells: elsewhere every flag sum is zero.
    const int cc = inb ? tid : p.nc - 1 - c0;  // in the tile
    const int S = (p.scnt + c0)[cc], C = inb ? (int)(p.ccnt + c0)[cc] : 0;
    const int8_t own = (p.smooth + c0)[cc];
    const int limited = (p.tlim + c0)[cc];
    // A wavefront's cells are one slice of the slot arrays; slot_face has a slice
    // of no slots for the wavefronts of the last tile past the last cell.
    const size_t slot0 = (size_t)((unsigned)(c0 + 64 * __builtin_amdgcn_readfirstlane(tid >> 6)) >> 6) * maxC * 64;
    const unsigned cl = tid & 63;
    int sfs[PF];
#pragma unroll
    for (int fi = 0; fi < PF; ++fi) sfs[fi] = fi < maxC ? (p.slot_face + slot0 + fi * 64)[cl] : 0;
    const int n16 = sten_words(tile, TILE, p.nc, p.stenW);
    const uint4* stSrc = reinterpret_cast<const uint4*>(p.sten + (size_t)tile * TILE * p.stenW);
    const int hn = p.hfix;
    const int32_t* hrow = p.halo + (size_t)tile * hn;
    const unsigned hid0 = (unsigned)hrow[min(tid, hn - 1)];
    const unsigned hid1 = (unsigned)hrow[min(tid + TILE, hn - 1)];
    const int m0 = p.more_ptr[tile], m1 = p.more_ptr[tile + 1];
    const int8_t hs0 = p.smooth[hid0];
    const int8_t hs1 = p.smooth[hid1];
    // A face's test counts only in a limited cell (the limiter condition, or
    // a flagged extended stencil, known after the flag sums): the
    // temperatures are requested here for cells meeting the condition and,
    // after the sums, for the others that turn out limited.  (Requesting
    // them in a flagged tile for every cell, with the stencil block, measured
    // slower.)
    R tfo[PF], tfn[PF], tvd[PF];
    unsigned short sks[PF];  // the face's flags of flat sides (DevPtrs::fflat)
    auto load_temps = [&](int fi) {
        const int sf = sfs[fi];
        const int f = (sf < 0 ? -sf : sf) - 1;
        if (fi < C && f < nf) {
            tfo[fi] = p.fvT[2 * f];
            tfn[fi] = p.fvT[2 * f + 1];
            tvd[fi] = (p.tTVD + slot0 + fi * 64)[cl];
            if (FLAT) sks[fi] = reinterpret_cast<const unsigned short*>(p.fflat)[f];
        }
    };
#pragma unroll
    for (int fi = 0; fi < PF; ++fi) {
        tfo[fi] = tfn[fi] = tvd[fi] = (R)0;
        sks[fi] = 0;
        if (limited) load_temps(fi);
    }
    if (inb) sS[tid] = own;
    if (tid < hn) sS[TILE + tid] = hs0;
    if (tid + TILE < hn) sS[2 * TILE + tid] = hs1;
    int flagged = (inb && own != 0) || (tid < hn && hs0 != 0) || (tid + TILE < hn && hs1 != 0);
    auto stage = [&](int j, int id) {
        const int8_t h = p.smooth[id];
        sS[j] = h;
        flagged |= h != 0;
    };
    for (int i = tid + 2 * TILE; i < hn; i += TILE) stage(TILE + i, hrow[i]);
    for (int i = m0 + tid; i < m1; i += TILE) stage(TILE + hn + i - m0, p.halo_more[i]);
    if (tid == 0) sS[TILE + p.hcap] = 0;  // the dummy member's flag
    int8_t shockType = own;
    int8_t shockTypeExt = own;
    // block-uniform: one wavefront's vote, or a workgroup reduction
    const bool anyFlagged = TILE == 64 ? __any(flagged) != 0 : __syncthreads_or(flagged) != 0;
    if (anyFlagged) {
        uint4* stDst = reinterpret_cast<uint4*>(sSt);
        const uint4 st0 = stSrc[min(tid, n16 - 1)];
        const uint4 st1 = stSrc[min(tid + TILE, n16 - 1)];
        const uint4 st2 = stSrc[min(tid + 2 * TILE, n16 - 1)];
        if (tid < n16) stDst[tid] = st0;
        if (tid + TILE < n16) stDst[tid + TILE] = st1;
        if (tid + 2 * TILE < n16) stDst[tid + 2 * TILE] = st2;
        for (int i = tid + 3 * TILE; i < n16; i += TILE) stDst[i] = stSrc[i];
        __syncthreads();
        if (inb) {
            // eight members to a 16-byte word of the cell's row; past its
            // stencil the row names the dummy member, whose flag is 0
            const uint4* row = reinterpret_cast<const uint4*>(sSt + tid * p.stenW);
            for (int ci = 0; ci < S; ci += 8) {
                const uint4 q = row[ci >> 3];
                const unsigned ids[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int8_t h = sS[(i & 1) ? ids[i >> 1] >> 16 : ids[i >> 1] & 0xffffu];
                    if (ci + i < C) shockType += h;
                    shockTypeExt += h;
                }
            }
        }
    }
    if (!inb) return;

    // Every face is visited; the reference leaves the loop at a cell's second
    // boundary face with bvd = 1, the largest value, so the result is the same.
    // cudaLimiter.h:431-448, with Tf_cur_TVD = Tc + BJ(lim) * (grad T . d) and
    // the condition lim < VALID_LIM_FACTOR taken from the reconstruction.
    int bvd = 0, bfaces = 0;
    const int isLimited = limited + (shockTypeExt > 0);
    if (isLimited && !limited) {
#pragma unroll
        for (int fi = 0; fi < PF; ++fi) load_temps(fi);
    }
    // The temperatures of a flat side, which are not stored, with the
    // reconstruction's operations: seldom a limited cell's own, more often its
    // neighbour's.
    auto form_flat = [&](int sf, unsigned sk, R& TfOwn, R& TfNei, R& Tf_cur_TVD) {
        const int f = (sf < 0 ? -sf : sf) - 1;
        const int2 oc = p.fcell[f];
        const double2 fc = p.fcen[f], fs = p.fshift ? p.fshift[f] : double2{0.0, 0.0};
        auto form = [&](bool nei, R& Tf) {
            const int s = nei ? oc.y : oc.x;
            const double2 cs = p.cen[s];
            const typename VT<R>::v2 g = p.gT[s];
            const R T = p.W[s].w;
            const R dx = (R)(fc.x - (nei ? cs.x + fs.x : cs.x)), dy = (R)(fc.y - (nei ? cs.y + fs.y : cs.y));
            Tf = T + g.x * dx + g.y * dy;
            if (nei == sf < 0) Tf_cur_TVD = T + (g.x * dx + g.y * dy);
        };
        if (sk & 0xff) form(false, TfOwn);
        if (sk >> 8) form(true, TfNei);
    };
    if (FLAT && __builtin_expect((sks[0] | sks[1] | sks[2] | sks[3]) != 0, 0)) {
        static_assert(PF == 4, "the flags of all slots read ahead");
#pragma unroll
        for (int fi = 0; fi < PF; ++fi)
            if (sks[fi]) form_flat(sfs[fi], sks[fi], tfo[fi], tfn[fi], tvd[fi]);
    }
    auto face = [&](int sf, R TfOwn, R TfNei, R Tf_cur_TVD) {
        const int isNei = sf < 0;
        const R Tf_cur = (R)isNei * TfNei + (R)(1 - isNei) * TfOwn;
        const R Tf_nei = (R)(1 - isNei) * TfNei + (R)isNei * TfOwn;
        const int typeval = fabs(Tf_cur_TVD - Tf_nei) < K<R>::BVD_FACTOR * fabs(Tf_cur - Tf_nei);
        const int isNotFlat = fabs(Tf_cur - Tf_nei) > K<R>::VSMALL;
        bvd = max(bvd, isNotFlat * isLimited * typeval);
    };
#pragma unroll
    for (int fi = 0; fi < PF; ++fi) {
        if (fi < C) {
            const int sf = sfs[fi];
            const int f = (sf < 0 ? -sf : sf) - 1;
            if (f >= nf)
                bfaces += 1;
            else if (isLimited)
                face(sf, tfo[fi], tfn[fi], tvd[fi]);
        }
    }
    for (int fi = PF; fi < C; ++fi) {  // cells with more than PF faces
        const int sf = (p.slot_face + slot0 + fi * 64)[cl];
        const int f = (sf < 0 ? -sf : sf) - 1;
        if (f >= nf)
            bfaces += 1;
        else if (isLimited) {
            R To = p.fvT[2 * f], Tn = p.fvT[2 * f + 1], Tt = (p.tTVD + slot0 + fi * 64)[cl];
            const unsigned sk = FLAT ? reinterpret_cast<const unsigned short*>(p.fflat)[f] : 0;
            if (FLAT && sk) form_flat(sf, sk, To, Tn, Tt);
            face(sf, To, Tn, Tt);
        }
    }
    if (bfaces >= 2) bvd = 1;  // corner cells use the second-order reconstruction
    int finalType = (shockType > 0) * (shockTypeExt > 1) * (-2) + (bvd > 0);
    if (p.boundaryFirstOrder && bfaces > 0) {
        // extension: a cell with a boundary face takes the first-order state
        // on its faces (TVD with zero limiter), generalising the reference's
        // corner-cell rule; shock types keep their flux choice.  A raw
        // limiter is never negative, so -1 marks the zero limiter.
        finalType = finalType ? finalType : 1;
        (p.ftype + c0)[tid] = (int8_t)finalType;
        p.lim[c] = v4{(R)-1, (R)-1, (R)-1, (R)-1};
        return;
    }
    // The limiter transform (cudaLimiter.h:453-461) is applied where the
    // limiter is used, by the face pass, from this type and the raw limiter:
    // the same function of the same values, without a write of the array.
    (p.ftype + c0)[tid] = (int8_t)finalType;
}

// The limiter the face pass uses: the transform of K6 applied to the raw K5
// limiter with the cell's final type, or zero for a first-order cell.  The
// reference blends both transforms, isShock * venkat + (1 - isShock) * bj
// (cudaLimiter.h:453-461); only the selected one is evaluated here, so that a
// wavefront without shock cells skips the Venkatakrishnan divisions.  The
// value is the blend's bit for bit: both transforms of a raw limiter >= 0 are
// finite (fmin(., 1) of a finite or NaN value), the Venkatakrishnan value is
// positive, and adding zero turns a BJ value of -0, where the blend gives
// +0 + -0 = +0, into +0.
// The four limiters of a side are transformed together, so that the divisions
// of a shock side run side by side.
template <typename R>
__device__ __forceinline__ typename VT<R>::v4 face_limiters(const typename VT<R>::v4& raw, int isShock) {
    R y[4] = {raw.x, raw.y, raw.z, raw.w}, t[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) t[i] = to_bj(y[i]);
    if (isShock) {
#pragma unroll
        for (int i = 0; i < 4; ++i) t[i] = to_venkat(y[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) t[i] = y[i] < (R)0 ? (R)0 : t[i] + (R)0;
    return {t[0], t[1], t[2], t[3]};
}

// ---------------------------------------------------------------- K7 flux

template <typename R>
__device__ __forceinline__ R minimize_delta(R L, R Rv, R LT, R RT) {
    // cudaRiemannSolver.h:7-14
    R d = fabs(Rv - L);
    d = fmin(d, fabs(Rv - LT));
    d = fmin(d, fabs(RT - L));
    d = fmin(d, fabs(RT - LT));
    return (R)(Rv >= L) * d - (R)(Rv < L) * d;
}

template <typename R>
__device__ __forceinline__ void kfvs_flux(R& rhoFlux, R& rhoUxFlux, R& rhoUyFlux, R& rhoEFlux, R rhoL, R rhoR,
                                          R pL, R pR, R uxL, R uxR, R uyL, R uyR, R TL, R TR, R Kd, R Cv, R magSf,
                                          R Sfx, R Sfy) {
    // cudaRiemannSolver.h:16-68
    const R nfx = Sfx / magSf, nfy = Sfy / magSf;
    const R uxLl = uxL * nfx + uyL * nfy, uyLl = uyL * nfx - uxL * nfy;
    const R uxRl = uxR * nfx + uyR * nfy, uyRl = uyR * nfx - uxR * nfy;
    const R lamL = (R)0.5 * rhoL / pL, lamR = (R)0.5 * rhoR / pR;
    const R PI = (R)3.141593;
    R erf[2], gauss[2];
    erfc_exp({-sqrt(lamL) * uxLl, sqrt(lamR) * uxRl}, {-lamL * uxLl * uxLl, -lamR * uxRl * uxRl}, erf, gauss);
    const R Mu0p = (R)0.5 * erf[0];
    const R Mu1p = uxLl * Mu0p + (R)0.5 * gauss[0] / (sqrt(PI * lamL));
    const R Mu2p = uxLl * Mu1p + (R)0.5 * Mu0p / lamL;
    const R Mu3p = uxLl * Mu2p + Mu1p / lamL;
    const R Mu0n = (R)0.5 * erf[1];
    const R Mu1n = uxRl * Mu0n - (R)0.5 * gauss[1] / (sqrt(PI * lamR));
    const R Mu2n = uxRl * Mu1n + (R)0.5 * Mu0n / lamR;
    const R Mu3n = uxRl * Mu2n + Mu1n / lamR;
    const R Mv1L = uyLl, Mv1R = uyRl;
    const R trho = rhoL * Mu1p + rhoR * Mu1n;
    const R trhoUx = rhoL * Mu2p + rhoR * Mu2n;
    const R trhoUy = rhoL * Mu1p * Mv1L + rhoR * Mu1n * Mv1R;
    const R trhoE = (R)0.5 * rhoL * (Mu3p + Mu1p * (uyLl * Mv1L + (R)0.5 / lamL) + Mu1p * Kd * (R)0.5 / lamL) +
                    (R)0.5 * rhoR * (Mu3n + Mu1n * (uyRl * Mv1R + (R)0.5 / lamR) + Mu1n * Kd * (R)0.5 / lamR);
    rhoUxFlux += trhoUx * Sfx - trhoUy * Sfy - (R)0.5 * (rhoFlux * uxL + pL * Sfx) - (R)0.5 * (rhoFlux * uxR + pR * Sfx);
    rhoUyFlux += trhoUx * Sfy + trhoUy * Sfx - (R)0.5 * (rhoFlux * uyL + pL * Sfy) - (R)0.5 * (rhoFlux * uyR + pR * Sfy);
    rhoEFlux += trhoE * magSf - (R)0.5 * rhoFlux * (Cv * TL + (R)0.5 * (uxL * uxL + uyL * uyL) + pL / rhoL) -
                (R)0.5 * rhoFlux * (Cv * TR + (R)0.5 * (uxR * uxR + uyR * uyR) + pR / rhoR);
    rhoFlux += trho * magSf - (R)0.5 * rhoL * (uxL * Sfx + uyL * Sfy) - (R)0.5 * rhoR * (uxR * Sfx + uyR * Sfy);
}

template <typename R>
__device__ __forceinline__ void roe_flux(R& rhoFlux, R& rhoUxFlux, R& rhoUyFlux, R& rhoEFlux, R rhoL, R rhoR, R pL,
                                         R pR, R uxL, R uxR, R uyL, R uyR, R TL, R TR, R dP, R dRho, R gamma, R Cv,
                                         R magSf, R Sfx, R Sfy) {
    // cudaRiemannSolver.h:71-136
    const R nfx = Sfx / magSf, nfy = Sfy / magSf;
    const R VL = uxL * nfx + uyL * nfy, VR = uxR * nfx + uyR * nfy;
    const R hL = Cv * TL + (R)0.5 * (uxL * uxL + uyL * uyL) + pL / rhoL;
    const R hR = Cv * TR + (R)0.5 * (uxR * uxR + uyR * uyR) + pR / rhoR;
    const R rhoT = sqrt(fmax(rhoL * rhoR, (R)1e-20));
    const R wL = sqrt(fmax(rhoL, (R)1e-20)) / (sqrt(fmax(rhoL, (R)1e-20)) + sqrt(fmax(rhoR, (R)1e-20)));
    const R wR = (R)1 - wL;
    const R uxT = uxL * wL + uxR * wR, uyT = uyL * wL + uyR * wR, hT = hL * wL + hR * wR;
    const R q2 = uxT * uxT + uyT * uyT;
    const R cT = sqrt(fmax((gamma - (R)1) * (hT - (R)0.5 * q2), (R)1e-20));
    const R VT_ = uxT * nfx + uyT * nfy;
    const R dUx = uxR - uxL, dUy = uyR - uyL;
    const R dV = dUx * nfx + dUy * nfy;
    const R r1 = (dP - rhoT * cT * dV) / ((R)2 * cT * cT);
    const R r2 = dRho - dP / (cT * cT);
    const R r3 = (dP + rhoT * cT * dV) / ((R)2 * cT * cT);
    const R cL = sqrt(fmax((gamma - (R)1) * (hL - (R)0.5 * (uxL * uxL + uyL * uyL)), (R)1e-20));
    const R cR = sqrt(fmax((gamma - (R)1) * (hR - (R)0.5 * (uxR * uxR + uyR * uyR)), (R)1e-20));
    // Harten's entropy fix, (l^2 + eps^2) / (2 eps + 1e-30) below eps.  At or
    // above eps the reference's blend, 1 * l + 0 * quotient, is l itself as
    // long as the quotient is finite, which it is below kMax (0 <= eps <= l):
    // the three divisions are left to wavefronts with a face that needs one
    // (of 17 on a Roe face; 740k cells in float 34.5 -> 32.5 us).
    constexpr R kMax = sizeof(R) == 8 ? (R)1e100 : (R)1e4;
    const R e1 = (R)2 * fmax((R)0, (VR - cR) - (VL - cL)), e2 = (R)2 * fmax((R)0, VR - VL),
            e3 = (R)2 * fmax((R)0, (VR + cR) - (VL + cL));
    R l1 = fabs(VT_ - cT), l2 = fabs(VT_), l3 = fabs(VT_ + cT);
    if (!(l1 >= e1 && l2 >= e2 && l3 >= e3 && fmax(l1, l3) < kMax)) {
        auto fix = [](R l, R e) {
            return (R)(l >= e) * l + (R)(l < e) * ((l * l + e * e) / ((R)2 * e + (R)1e-30));
        };
        l1 = fix(l1, e1);
        l2 = fix(l2, e2);
        l3 = fix(l3, e3);
    }
    rhoFlux -= (R)0.5 * (l1 * r1 + l2 * r2 + l3 * r3) * magSf;
    rhoUxFlux -= (R)0.5 * (l1 * r1 * (uxT - cT * nfx) + l2 * (r2 * uxT + rhoT * (dUx - dV * nfx)) + l3 * r3 * (uxT + cT * nfx)) * magSf;
    rhoUyFlux -= (R)0.5 * (l1 * r1 * (uyT - cT * nfy) + l2 * (r2 * uyT + rhoT * (dUy - dV * nfy)) + l3 * r3 * (uyT + cT * nfy)) * magSf;
    rhoEFlux -= (R)0.5 * (l1 * r1 * (hT - cT * VT_) + l2 * (r2 * (R)0.5 * q2 + rhoT * (uxT * dUx + uyT * dUy - VT_ * dV)) +
                          l3 * r3 * (hT + cT * VT_)) * magSf;
}

// Waves per SIMD the register allocator must allow for the face-centre flux
// pass, per working type (build-time tuning knobs; 1 = no constraint).  The
// FP64 passes take 128 VGPRs (4 waves) unconstrained, the float ones 63 and 70
// (8 and 7 waves).  The FP64 pass with the CFL bound took 136 (3 waves) and 135
// us on 1.5M cells while it formed the bound's distances itself; with them
// stored, the gas constants from the host and the bound kept in LDS it has 4
// waves: 120 us (without the bound 113 -> 108, entropy fix below).  At 5 waves
// 44 and 61 VGPRs spill.
#ifndef AFAR_FLUX_WPE_D
#define AFAR_FLUX_WPE_D 1
#endif
#ifndef AFAR_FLUX_DT_WPE_D
#define AFAR_FLUX_DT_WPE_D 1
#endif
#ifndef AFAR_FLUX_WPE_F
#define AFAR_FLUX_WPE_F 1
#endif
template <typename R, bool DT, bool GP> struct FluxWaves {
    static constexpr int value =
        GP ? 1 : (sizeof(R) == 8 ? (DT ? AFAR_FLUX_DT_WPE_D : AFAR_FLUX_WPE_D) : AFAR_FLUX_WPE_F);
};

// DT: also reduce the CFL bound of every internal face to one partial minimum
// per block (dt_part[blockIdx.x]); the bound is a function of the
// primitive state alone, which no kernel of the stage has changed yet.
template <typename R, bool DT, bool GP, int B = 256>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(FluxWaves<R, DT, GP>::value, 8))) void k_flux(
    DevPtrs<R> p, GasArgs gas) {
    using v4 = typename VT<R>::v4;
    using v2 = typename VT<R>::v2;
    constexpr bool FLAT = FormsFlat<R, GP>::value;
    const int tile = xcd_tile(p.map);
    if (tile < 0) return;
    static_assert(!DT || B == 256, "a partial per 256 faces");
    const int i = tile * B + threadIdx.x;
    const int nf = p.nf;
    // each face's bound waits in LDS for the reduction at the end: two
    // registers fewer through the flux, which has none to spare for its waves
    __shared__ double sDt[DT ? 256 : 1];
    if (DT) sDt[threadIdx.x] = 1e5;
    if (i < nf) {
        const int f = i;
        const int2 oc = p.fcell[f];
        const int own = oc.x, nei = oc.y;
        // sides whose face state and limiters are formed here (DevPtrs::fflat)
        bool skL = false, skR = false;
        if constexpr (FLAT) {
            const uchar2 sk = reinterpret_cast<const uchar2*>(p.fflat)[f];
            skL = sk.x != 0;
            skR = sk.y != 0;
        }
        // The face's area vector, in double where the CFL bound needs it, and
        // (at the face centre) its centre's offsets from the two cell centres:
        // FP64 forms them with the host layout's expressions, the neighbour's
        // centre shifted; FP32-mixed reads them rounded to float.
        R magSf, Sfx, Sfy, dxL = 0, dyL = 0, dxR = 0, dyR = 0;
        double2 sf{}, cg{};
        double mag = 0.0;
        if constexpr (sizeof(R) == 4 && !DT) {
            const float4 s = p.fsf32[f];
            Sfx = s.x;
            Sfy = s.y;
            magSf = s.z;
        } else {
            sf = p.fsf[f];
            mag = p.fmag[f];
            Sfx = (R)sf.x;
            Sfy = (R)sf.y;
            magSf = (R)mag;
        }
        if constexpr (DT) cg = p.fcfl[f];
        if constexpr (!GP && sizeof(R) == 4) {
            const float4 o = p.foff32[f];
            dxL = o.x;
            dyL = o.y;
            dxR = o.z;
            dyR = o.w;
        } else if constexpr (!GP) {
            const double2 fc = p.fcen[f], co = p.cen[own], cn = p.cen[nei];
            const double2 fs = p.fshift ? p.fshift[f] : double2{0.0, 0.0};
            dxL = (R)(fc.x - co.x);
            dyL = (R)(fc.y - co.y);
            dxR = (R)(fc.x - (cn.x + fs.x));
            dyR = (R)(fc.y - (cn.y + fs.y));
        }
        const int8_t to = p.ftype[own], tn = p.ftype[nei];
        const int isTVD_L = to != 0, isTVD_R = tn != 0;
        const int isShock = to < 0 || tn < 0;
        const R Rg = (R)gas.R;
        const v4 wL = p.W[own], wR = p.W[nei];
        const v2 gpL = p.gp[own], gTL = p.gT[own];
        const v2 gpR = p.gp[nei], gTR = p.gT[nei];
        // Raw limiters and face-centre O3 states of both sides.  A flat side
        // reads the entry of ones behind the cells' limiters, a face with two
        // of them face 0's states: no branches, and no memory traffic.
        const v4 rL = p.lim[FLAT && skL ? p.nc : own], rR = p.lim[FLAT && skR ? p.nc : nei];
        v4 fL0{}, fR0{};
        if constexpr (!GP) {
            if constexpr (sizeof(R) == 8) {  // one 2-vector per variable
                const int fr = skL && skR ? 0 : f;
                const v2 sp = reinterpret_cast<const v2*>(p.fvp)[fr], su = reinterpret_cast<const v2*>(p.fvu)[fr];
                const v2 sv = reinterpret_cast<const v2*>(p.fvv)[fr], sT = reinterpret_cast<const v2*>(p.fvT)[fr];
                fL0 = v4{sp.x, su.x, sv.x, sT.x};
                fR0 = v4{sp.y, su.y, sv.y, sT.y};
            } else {
                fL0 = p.fv[2 * f];
                fR0 = p.fv[2 * f + 1];
            }
        }
        if (DT) {
            const double d = cfl_face_dt(sf.x, sf.y, mag, cg, wL, wR, gas.c2T, gas.CFL);
            sDt[threadIdx.x] = d < 1e5 ? d : 1e5;
        }
        const int shL = to < 0, shR = tn < 0;
        const v4 lL = face_limiters<R>(rL, shL);
        const v4 lR = face_limiters<R>(rR, shR);
        // The limited linear velocities enter the flux only on a TVD side: on
        // an O3 side they are blended with weight 0, which adds a zero to the
        // O3 velocity, so they change nothing unless that velocity is itself a
        // zero (whose sign the added zero decides).  Their gradients are read
        // only where they can matter (at the face centre).  A non-finite
        // velocity gradient beside a finite O3 state (a degenerate
        // least-squares stencil) would turn that blend into NaN in the
        // reference; here it is not read.  A flat cell's state is linear and
        // takes them too; it is formed with the reconstruction's operations.
        v2 guL{}, gvL{}, guR{}, gvR{};
        if (GP || skL || isTVD_L || fL0.y == (R)0 || fL0.z == (R)0) {
            guL = p.gu[own];
            gvL = p.gv[own];
        }
        if (GP || skR || isTVD_R || fR0.y == (R)0 || fR0.z == (R)0) {
            guR = p.gu[nei];
            gvR = p.gv[nei];
        }
        if (FLAT && skL)
            fL0 = v4{wL.x + gpL.x * dxL + gpL.y * dyL, wL.y + guL.x * dxL + guL.y * dyL,
                     wL.z + gvL.x * dxL + gvL.y * dyL, wL.w + gTL.x * dxL + gTL.y * dyL};
        if (FLAT && skR)
            fR0 = v4{wR.x + gpR.x * dxR + gpR.y * dyR, wR.y + guR.x * dxR + guR.y * dyR,
                     wR.z + gvR.x * dxR + gvR.y * dyR, wR.w + gTR.x * dxR + gTR.y * dyR};

        // the flux of the two states reconstructed at a point with offsets
        // (dxL, dyL) from the owner and (dxR, dyR) from the neighbour; fL, fR
        // are the high-order (O3) states there
        auto point_flux = [&](R dxL, R dyL, R dxR, R dyR, const v4& fL, const v4& fR, R& out0, R& out1, R& out2,
                              R& out3) {
            const R pLT = wL.x + lL.x * (gpL.x * dxL + gpL.y * dyL);
            const R uxLT = wL.y + lL.y * (guL.x * dxL + guL.y * dyL);
            const R uyLT = wL.z + lL.z * (gvL.x * dxL + gvL.y * dyL);
            const R TLT = wL.w + lL.w * (gTL.x * dxL + gTL.y * dyL);
            const R rhoLT = pLT / (Rg * TLT);
            const R pRT = wR.x + lR.x * (gpR.x * dxR + gpR.y * dyR);
            const R uxRT = wR.y + lR.y * (guR.x * dxR + guR.y * dyR);
            const R uyRT = wR.z + lR.z * (gvR.x * dxR + gvR.y * dyR);
            const R TRT = wR.w + lR.w * (gTR.x * dxR + gTR.y * dyR);
            const R rhoRT = pRT / (Rg * TRT);

            const R pL = (R)(1 - isTVD_L) * fL.x + (R)isTVD_L * pLT;
            const R uxL = (R)(1 - isTVD_L) * fL.y + (R)isTVD_L * uxLT;
            const R uyL = (R)(1 - isTVD_L) * fL.z + (R)isTVD_L * uyLT;
            const R TL = (R)(1 - isTVD_L) * fL.w + (R)isTVD_L * TLT;
            const R rhoL = pL / (Rg * TL);
            const R pR = (R)(1 - isTVD_R) * fR.x + (R)isTVD_R * pRT;
            const R uxR = (R)(1 - isTVD_R) * fR.y + (R)isTVD_R * uxRT;
            const R uyR = (R)(1 - isTVD_R) * fR.z + (R)isTVD_R * uyRT;
            const R TR = (R)(1 - isTVD_R) * fR.w + (R)isTVD_R * TRT;
            const R rhoR = pR / (Rg * TR);

            const R dP = minimize_delta(pL, pR, pLT, pRT);
            const R dRho = minimize_delta(rhoL, rhoR, rhoLT, rhoRT);

            const R CvR = (R)gas.Cv;
            R rhoFlux = (R)0.5 * rhoL * (uxL * Sfx + uyL * Sfy) + (R)0.5 * rhoR * (uxR * Sfx + uyR * Sfy);
            R rhoUxFlux = (R)0.5 * (rhoFlux * uxL + pL * Sfx) + (R)0.5 * (rhoFlux * uxR + pR * Sfx);
            R rhoUyFlux = (R)0.5 * (rhoFlux * uyL + pL * Sfy) + (R)0.5 * (rhoFlux * uyR + pR * Sfy);
            R rhoEFlux = (R)0.5 * rhoFlux * (CvR * TL + (R)0.5 * (uxL * uxL + uyL * uyL) + pL / rhoL) +
                         (R)0.5 * rhoFlux * (CvR * TR + (R)0.5 * (uxR * uxR + uyR * uyR) + pR / rhoR);
            if (isShock)
                kfvs_flux<R>(rhoFlux, rhoUxFlux, rhoUyFlux, rhoEFlux, rhoL, rhoR, pL, pR, uxL, uxR, uyL, uyR, TL, TR,
                             (R)gas.Kd, CvR, magSf, Sfx, Sfy);
            else
                roe_flux<R>(rhoFlux, rhoUxFlux, rhoUyFlux, rhoEFlux, rhoL, rhoR, pL, pR, uxL, uxR, uyL, uyR, TL, TR, dP,
                            dRho, (R)gas.gamma, CvR, magSf, Sfx, Sfy);
            out0 = rhoFlux;
            out1 = rhoUxFlux;
            out2 = rhoUyFlux;
            out3 = rhoEFlux;
        };
        if constexpr (!GP) {
            R rhoFlux, rhoUxFlux, rhoUyFlux, rhoEFlux;
            point_flux(dxL, dyL, dxR, dyR, fL0, fR0, rhoFlux, rhoUxFlux, rhoUyFlux, rhoEFlux);
            if constexpr (sizeof(R) == 4)
                p.flux32[f] = float4{rhoFlux, rhoUxFlux, rhoUyFlux, rhoEFlux};
            else
                p.flux[f] = double4{(double)rhoFlux, (double)rhoUxFlux, (double)rhoUyFlux, (double)rhoEFlux};
        } else {
            // extension: weighted sum over the face's quadrature points
            double4 acc = double4{0.0, 0.0, 0.0, 0.0};
            for (int g = 0; g < p.ngp; ++g) {
                const v4 d = p.fgd[(size_t)g * nf + f];
                R rhoFlux, rhoUxFlux, rhoUyFlux, rhoEFlux;
                point_flux((R)d.x, (R)d.y, (R)d.z, (R)d.w, p.fvg[((size_t)g * nf + f) * 2],
                           p.fvg[((size_t)g * nf + f) * 2 + 1], rhoFlux, rhoUxFlux, rhoUyFlux, rhoEFlux);
                const double w = p.gpw[g];
                if (g == 0) {
                    acc = double4{w * (double)rhoFlux, w * (double)rhoUxFlux, w * (double)rhoUyFlux,
                                  w * (double)rhoEFlux};
                } else {
                    acc.x += w * (double)rhoFlux;
                    acc.y += w * (double)rhoUxFlux;
                    acc.z += w * (double)rhoUyFlux;
                    acc.w += w * (double)rhoEFlux;
                }
            }
            p.flux[f] = acc;
        }
    } else if (i < nf + p.nb) {
        // boundary faces: physical flux of the ghost state (cudaRiemannSolver.h:254-270)
        const int b = i - nf;
        const double4 g = p.bgeo[b];
        const typename VT<R>::v4 w = p.W[p.nc + b];
        const double bp = w.x, bUx = w.y, bUy = w.z, bT = w.w;
        const double rho = bp / (gas.R * bT);
        const double rhoFlux = rho * (bUx * g.x + bUy * g.y);
        p.flux[i] = double4{rhoFlux, rhoFlux * bUx + bp * g.x, rhoFlux * bUy + bp * g.y,
                            rhoFlux * (gas.Cv * bT + 0.5 * (bUx * bUx + bUy * bUy) + bp / rho)};
    }
    if (DT) {
        // Two partials per tile of 256 faces: slot 0 for the instance of the
        // tile's first face, slot 1 for the next one (every instance of a
        // batch has at least 256 internal faces, so a tile meets at most two).
        const int f0 = min(tile * 256, nf - 1);
        const int i0 = (p.cinst && nf > 0) ? p.cinst[p.fcell[f0].x] : 0;
        const int mine = (i < nf && p.cinst) ? p.cinst[p.fcell[i].x] : i0;
        __shared__ double wmin[4];
        const double dtf = sDt[threadIdx.x];
        const double m0 = block_min_256(mine == i0 ? dtf : 1e5, wmin);
        const double m1 = block_min_256(mine == i0 ? 1e5 : dtf, wmin);
        if (threadIdx.x == 0) {
            p.dt_part[2 * tile] = m0;
            p.dt_part[2 * tile + 1] = m1;
        }
    }
}

// Density residual norm: per block the sum over its cells of (Res_rho/V)^2
// (the residual gathered as in the update), then one block adds the partials
// in index order.  Fixed launch shapes make the sum order, and so the value,
// reproducible.
// The flux of face f (internal or boundary) as the residual gather reads it.
template <typename R> __device__ __forceinline__ double4 face_flux(const DevPtrs<R>& p, int f) {
    if (p.flux32 && f < p.nf) {
        const float4 q = p.flux32[f];
        return double4{(double)q.x, (double)q.y, (double)q.z, (double)q.w};
    }
    return p.flux[f];
}

template <typename R>
__global__ __launch_bounds__(256) void k_residual_part(DevPtrs<R> p) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    double v = 0.0;
    if (c < p.nc) {
        const int C = p.ccnt[c], maxC = p.maxC;
        double r0 = 0.0;
        for (int fi = 0; fi < C; ++fi) {
            const int sf = p.slot_face[sell(c, fi, maxC)];
            const int dir = (sf > 0) - (sf < 0);
            const int f = (sf < 0 ? -sf : sf) - 1;
            r0 += dir * face_flux(p, f).x;
        }
        const double q = r0 / p.vol[c];
        v = q * q;
    }
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    __shared__ double ws[4];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) p.res_part[blockIdx.x] = ((ws[0] + ws[1]) + ws[2]) + ws[3];
}

__global__ __launch_bounds__(1024) void k_residual_sum(const double* part, int n, double* out) {
    double v = 0.0;
    for (int i = threadIdx.x; i < n; i += 1024) v += part[i];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    __shared__ double ws[16];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < 16; ++w) s += ws[w];
        *out = s;
    }
}

// Time step of instance blockIdx.x: minimum of the flux kernel's partials
// over the tiles holding its internal faces (one block per instance).
__global__ __launch_bounds__(1024) void k_dt_reduce(double* dt, const double* part, const int32_t* finst_off,
                                                    double* tctl) {
    const int inst = blockIdx.x;
    const int fa = finst_off[inst], fb = finst_off[inst + 1];
    double v = 1e5;
    if (fb > fa) {
        const int t0 = fa >> 8, t1 = (fb - 1) >> 8;
        for (int t = t0 + (int)threadIdx.x; t <= t1; t += 1024) {
            const double o = part[2 * t + ((t == t0 && (fa & 255)) ? 1 : 0)];
            v = o < v ? o : v;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off);
        v = o < v ? o : v;
    }
    __shared__ double wmin[16];
    if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = wmin[0];
        for (int w = 1; w < 16; ++w) m = wmin[w] < m ? wmin[w] : m;
        // clip to the end time as the reference's caller does with
        // Foam::Time (dt = min(dt, t_end - t)); 0 once the end is reached
        double* tc = tctl + 4 * inst;
        const double t = tc[0], te = tc[1];
        double d = 0.0;
        if (t < te) {
            const double rem = te - t;
            d = m < rem ? m : rem;
            tc[0] = t + d;
            tc[2] += 1.0;  // steps taken
        }
        dt[inst] = d;
    }
}

// ---------------------------------------------------------------- K8-K11 update

__device__ __forceinline__ double4 boundary_value(int label, double4 w, double4 g, double4 val) {
    // src/CUDA/BCs/2D/*.h, dispatch table cudaEulerBCs.h:34-39; label 6 = per-patch fixed value
    switch (label) {
        case 0: return double4{w.x, 0.0, 0.0, 1.0};
        case 1: return double4{w.x, 0.0, 0.0, w.w};
        case 2: {
            const double nfx = g.x / g.z, nfy = g.y / g.z;
            return double4{w.x, w.y - (w.y * nfx + w.z * nfy) * nfx, w.z - (w.y * nfx + w.z * nfy) * nfy, w.w};
        }
        case 3: return double4{1.0, 3.0, 0.0, 1.0};
        case 4: return w;
        case 5: return double4{30.05945, 4.07795, 0.0, 5.97677};
        default: return val;
    }
}

__device__ __forceinline__ double4 primitive_state(const double4& u, double Rgas, double gamma) {
    const double pr = (gamma - 1.0) * (u.w - 0.5 * (u.y * u.y + u.z * u.z) / u.x);
    return double4{pr, u.y / u.x, u.z / u.x, pr / (Rgas * u.x)};
}

// Threads per block of the update, and of the flux pass without the CFL bound
// (whose tiles of 256 faces carry its partials): 64 where blocks of 256 would
// leave compute units without one, so that the waves' loads are issued from
// more of them.  20k quads 73.9 -> 72.7 us a step, FP32-mixed 67.1 -> 66.2, 17k
// periodic quads 59.9 -> 58.6, 800 quads 87.6 -> 84.8; 1.5M triangles with 64 everywhere 1110 -> 1113.
template <typename R, int B>
__global__ __launch_bounds__(B) void k_update(DevPtrs<R> p, double Rgas, double gamma, double dt_val,
                                                 const double* dt_ptr, double b1, double b2, double b3, int last) {
    const int tile = xcd_tile(p.map);
    if (tile < 0) return;
    const int c = tile * B + threadIdx.x;
    if (c >= p.nc) return;
    const int maxC = p.maxC, nf = p.nf;
    // Bound by its loads.  The first PF slots' faces are requested at once, then
    // their fluxes, so that a cell waits for two memory rounds and not for two
    // per face; a padding slot (0) reads face 0 and is left out of the sums.
    // Back to back on 1.5M cells 55.7 -> 48.1 us (FP64), 250k quads 12.9 ->
    // 10.8, 20k quads 5.2 -> 4.7 (a launch that only reduces 157 values takes 2.5).
    constexpr int PF = 4;
    int sfs[PF];
#pragma unroll
    for (int fi = 0; fi < PF; ++fi) sfs[fi] = fi < maxC ? p.slot_face[sell(c, fi, maxC)] : 0;
    const int C = p.ccnt[c];
    const double V = p.vol[c];
    // b2 = 0 (first stage): U equals Uold at the start of every step (both
    // are stored from one value at the end of a step and at upload), so the
    // stage reads it once; b2 * u is then b2 * uo, the same value
    const double4 uo = p.Uold[c], u = b2 == 0.0 ? uo : p.U[c];
    const double dt = dt_ptr ? dt_ptr[p.cinst ? p.cinst[c] : 0] : dt_val;
    double4 F[PF];
#pragma unroll
    for (int fi = 0; fi < PF; ++fi) {
        const int f = max((sfs[fi] < 0 ? -sfs[fi] : sfs[fi]) - 1, 0);
        F[fi] = face_flux(p, f);
    }
    if (dt_ptr && dt == 0.0) return;  // device path past its end time: the state stays
    double r0 = 0.0, r1 = 0.0, r2 = 0.0, r3 = 0.0;
    auto add = [&](int sf, const double4& Fs) {
        const int dir = (sf > 0) - (sf < 0);
        r0 += dir * Fs.x;
        r1 += dir * Fs.y;
        r2 += dir * Fs.z;
        r3 += dir * Fs.w;
    };
#pragma unroll
    for (int fi = 0; fi < PF; ++fi)
        if (sfs[fi] != 0) add(sfs[fi], F[fi]);
    for (int fi = PF; fi < C; ++fi) {
        const int sf = p.slot_face[sell(c, fi, maxC)];
        add(sf, face_flux(p, (sf < 0 ? -sf : sf) - 1));
    }
    const double rho = b1 * uo.x + b2 * u.x + b3 * dt * (-r0 / V);
    const double rhoUx = b1 * uo.y + b2 * u.y + b3 * dt * (-r1 / V);
    const double rhoUy = b1 * uo.z + b2 * u.z + b3 * dt * (-r2 / V);
    const double rhoE = b1 * uo.w + b2 * u.w + b3 * dt * (-r3 / V);
    const double4 un = double4{rho, rhoUx, rhoUy, rhoE};
    // The last stage's result is the next step's starting state, which the
    // next first stage reads from Uold alone; U would only be overwritten by
    // that stage, so it is not written here (the host reads the state from
    // Uold after a full step).
    if (last)
        p.Uold[c] = un;
    else
        p.U[c] = un;
    const double4 w = primitive_state(un, Rgas, gamma);
    typename VT<R>::v4 wr;
    wr.x = (R)w.x;
    wr.y = (R)w.y;
    wr.z = (R)w.z;
    wr.w = (R)w.w;
    p.W[c] = wr;
    // ghost states of this cell's boundary faces (K10), from the updated state
    auto ghost = [&](int sf) {
        const int f = sf - 1;
        if (f < nf) return;
        const int b = f - nf;
        const double4 g = boundary_value(p.blabel[b], w, p.bgeo[b], p.bval[b]);
        typename VT<R>::v4 gr;
        gr.x = (R)g.x;
        gr.y = (R)g.y;
        gr.z = (R)g.z;
        gr.w = (R)g.w;
        p.W[p.nc + b] = gr;
    };
#pragma unroll
    for (int fi = 0; fi < PF; ++fi) ghost(sfs[fi]);
    for (int fi = PF; fi < C; ++fi) ghost(p.slot_face[sell(c, fi, maxC)]);
}

// ---------------------------------------------------------------- output

// Rows idx[0..n) of the conserved state, in that order.  In the host's hands
// the same took a copy, two permutations and two temporary arrays: 12 ms for
// 1.5M cells (now 2-3, bound by the copy to pageable memory), 4 ms for 24
// batched meshes.
__global__ __launch_bounds__(256) void k_gather_state(const double4* src, const int32_t* idx, double4* dst, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[idx[i]];
}

// Rows idx[0..n) of the primitive state as doubles and of the flags: the
// types, or with pairs (smoothness flag, type) each.
template <typename R>
__global__ __launch_bounds__(256) void k_gather_fields(DevPtrs<R> p, const int32_t* idx, double4* W, int8_t* flags,
                                                       int pairs, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int c = idx[i];
    const typename VT<R>::v4 w = p.W[c];
    W[i] = double4{(double)w.x, (double)w.y, (double)w.z, (double)w.w};
    if (pairs) {
        flags[2 * i] = p.smooth[c];
        flags[2 * i + 1] = p.ftype[c];
    } else {
        flags[i] = p.ftype[c];
    }
}

// The face states and limiters that the last FP64 face-centre reconstruction
// left out, for a caller that fetches them.  It started from U where a full step
// followed it (the second stage's result: the third writes Uold), and from W
// where none did, or where the step's device time step was 0.
__global__ __launch_bounds__(256) void k_store_flat(DevPtrs<double> p, const double4* U, const double* dt_ptr,
                                                    double Rgas, double gamma) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= p.nc || !p.flat_prev[c]) return;
    const int C = p.ccnt[c], maxC = p.maxC, nf = p.nf;
    if (p.boundaryFirstOrder)  // cells with a boundary face were stored
        for (int fi = 0; fi < C; ++fi)
            if (abs(p.slot_face[sell(c, fi, maxC)]) - 1 >= nf) return;
    const bool stepped = U && !(dt_ptr && dt_ptr[p.cinst ? p.cinst[c] : 0] == 0.0);
    const double4 w = stepped ? primitive_state(U[c], Rgas, gamma) : p.W[c];
    const double2 gp = p.gp[c], gu = p.gu[c], gv = p.gv[c], gT = p.gT[c];
    p.lim[c] = double4{1.0, 1.0, 1.0, 1.0};
    for (int fi = 0; fi < C; ++fi) {
        const int sf = p.slot_face[sell(c, fi, maxC)];
        const int f = (sf < 0 ? -sf : sf) - 1;
        if (f >= nf) continue;
        const double2 d = p.slot_d[sell(c, fi, maxC)];
        store_face_state(p, 2 * f + (sf < 0),
                         double4{w.x + gp.x * d.x + gp.y * d.y, w.y + gu.x * d.x + gu.y * d.y,
                                 w.z + gv.x * d.x + gv.y * d.y, w.w + gT.x * d.x + gT.y * d.y});
    }
}

// ---------------------------------------------------------------- launchers

void launch_store_flat(const DevPtrs<double>& p, const double4* U, const double* dt_ptr, double Rg, double gamma,
                       hipStream_t s) {
    hipLaunchKernelGGL(k_store_flat, dim3((p.nc + 255) / 256), dim3(256), 0, s, p, U, dt_ptr, Rg, gamma);
}

void launch_gather_state(const double4* src, const int32_t* idx, double4* dst, int n, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_gather_state, dim3((n + 255) / 256), dim3(256), 0, s, src, idx, dst, n);
}

template <typename R>
void launch_gather_fields(const DevPtrs<R>& p, const int32_t* idx, double4* W, int8_t* flags, int pairs, int n,
                          hipStream_t s) {
    if (n > 0)
        hipLaunchKernelGGL(k_gather_fields<R>, dim3((n + 255) / 256), dim3(256), 0, s, p, idx, W, flags, pairs, n);
}

template <typename R>
void launch_lsq(const DevPtrs<R>& p, hipStream_t s) {
    if (p.nc == 0) return;
    hipLaunchKernelGGL(k_lsq<R>, dim3((p.nc + 255) / 256), dim3(256), 0, s, p);
}

// p with the map of a kernel of n tiles and its grid: a block per tile, rounded
// up to chunks of equal size.  maxLog: the most chunks (the CFL pass, whose
// partials and tickets count the grid's blocks).
// 8 chunks at least, 128 at most, and between them the most that leave each
// 2048 cells (FP64) or 4096 (FP32-mixed, half the bytes): smaller chunks leave
// the XCDs evenly loaded where the flow is flat in part of the mesh (eighths:
// 65k quads of a corner flow 102 -> 112 us a step, 260k 197 -> 228), more of
// them than 128 break up the streams of the largest meshes (1.5M triangles
// 1131 us with 128, 1154 with 512; with eighths 1237).  Past 128 a chunk holds
// at most 12288 cells: 256 FP32-mixed corner flows, 8.2M cells in the largest
// bucket, 7.54 -> 7.41 ms a step; triangles and quads with 128 chunks and so, FP64:
// 1.7M cells 978 -> 956 us, 2.3M 1318 -> 1298, 3.8M 2095 -> 2100, 6.6M 3528 -> 3453,
// FP32-mixed: 965 -> 957, 1325 -> 1316, 2129 -> 2083, 3622 -> 3531.
template <typename R>
static DevPtrs<R> mapped(const DevPtrs<R>& p, int n, unsigned& grid, int maxLog = 24) {
    constexpr int kChunkCells = 16384 / sizeof(R), kMaxChunkCells = 12288;
    int mlog = 3;
    while (mlog < 7 && p.nc >> (mlog + 1) >= kChunkCells) ++mlog;
    while (mlog < maxLog && p.nc >> mlog > kMaxChunkCells) ++mlog;
    while (mlog < maxLog && ((unsigned long long)n * n) >> (mlog + 3) >= 1ull << 31) ++mlog;  // keeps i * per below 2^32
    DevPtrs<R> q = p;
    const unsigned per = std::max(1u, ((unsigned)n + (1u << mlog) - 1) >> mlog);
    q.map = TileMap{n, (int)per, mlog, per == 1 ? 0u : 0xffffffffu / per + 1u};
    grid = per << mlog;
    return q;
}

template <typename R>
void launch_cfl(const DevPtrs<R>& p, double Rg, double Cv, double CFL, double* host_dt, hipStream_t s) {
    const int nt = std::min(kCflBlocks, std::max(1, (p.nf + 255) / 256));
    const int chunk = (p.nf + nt - 1) / nt;
    unsigned grid;
    static_assert(kCflBlocks == 1 << 10, "a tile per block and no more chunks than blocks");
    const DevPtrs<R> q = mapped(p, nt, grid, 10);
    hipLaunchKernelGGL(k_cfl<R>, dim3(grid), dim3(256), 0, s, q, gas_args<R>(Rg, Cv, CFL).c2T, CFL, chunk, host_dt);
}

template <typename R, bool GP, int MS>
void launch_reconstruct_q(const DevPtrs<R>& p, int nb, int tile, size_t lds, hipStream_t s) {
    switch (tile) {
        case 64: hipLaunchKernelGGL((k_reconstruct_q<R, 64, GP, MS>), dim3(nb), dim3(256), lds, s, p); break;
        case 128: hipLaunchKernelGGL((k_reconstruct_q<R, 128, GP, MS>), dim3(nb), dim3(512), lds, s, p); break;
        default: hipLaunchKernelGGL((k_reconstruct_q<R, 256, GP, MS>), dim3(nb), dim3(1024), lds, s, p); break;
    }
}

template <typename R, bool GP>
void launch_reconstruct_t(const DevPtrs<R>& p, int nb, int tile, size_t lds, hipStream_t s, int lanes) {
    if (lanes == 4) {
        if (p.maxS <= 8)
            launch_reconstruct_q<R, GP, 8>(p, nb, tile, lds, s);
        else if (p.maxS <= 16)
            launch_reconstruct_q<R, GP, 16>(p, nb, tile, lds, s);
        else
            launch_reconstruct_q<R, GP, kMaxSten>(p, nb, tile, lds, s);
        return;
    }
    switch (tile) {
        case 64: hipLaunchKernelGGL((k_reconstruct<R, 64, GP>), dim3(nb), dim3(64), lds, s, p); break;
        case 128: hipLaunchKernelGGL((k_reconstruct<R, 128, GP>), dim3(nb), dim3(128), lds, s, p); break;
        default: hipLaunchKernelGGL((k_reconstruct<R, 256, GP>), dim3(nb), dim3(256), lds, s, p); break;
    }
}

template <typename R>
void launch_reconstruct(const DevPtrs<R>& dev, int tile, size_t lds, hipStream_t s, int lanes) {
    unsigned nb;
    const DevPtrs<R> p = mapped(dev, dev.ntiles, nb);
    if (p.ngp > 0) {
        launch_reconstruct_t<R, true>(p, nb, tile, lds, s, lanes);
        return;
    }
    launch_reconstruct_t<R, false>(p, nb, tile, lds, s, lanes);
}

template <typename R>
void launch_bvd(const DevPtrs<R>& dev, int tile, size_t lds, hipStream_t s) {
    unsigned nb;
    const DevPtrs<R> p = mapped(dev, dev.ntiles, nb);
    switch (tile) {
        case 64: hipLaunchKernelGGL((k_bvd<R, 64>), dim3(nb), dim3(64), lds, s, p); break;
        case 128: hipLaunchKernelGGL((k_bvd<R, 128>), dim3(nb), dim3(128), lds, s, p); break;
        default: hipLaunchKernelGGL((k_bvd<R, 256>), dim3(nb), dim3(256), lds, s, p); break;
    }
}

// Whether n threads in blocks of 256 are no more blocks than the chip has CUs (256).
static bool small_blocks(int n) { return n <= 256 * 256; }

int flux_tiles(int nf, int nb) { return std::max(1, (nf + nb + 255) / 256); }

template <typename R>
void launch_flux(const DevPtrs<R>& dev, double Rg, double Cv, hipStream_t s) {
    unsigned grid;
    const int n = dev.nf + dev.nb, B = small_blocks(n) ? 64 : 256;
    const DevPtrs<R> p = mapped(dev, std::max(1, (n + B - 1) / B), grid);
    const GasArgs gas = gas_args<R>(Rg, Cv, 0.0);
    if (p.ngp > 0)
        hipLaunchKernelGGL((B == 64 ? k_flux<R, false, true, 64> : k_flux<R, false, true, 256>), dim3(grid), dim3(B), 0,
                           s, p, gas);
    else
        hipLaunchKernelGGL((B == 64 ? k_flux<R, false, false, 64> : k_flux<R, false, false, 256>), dim3(grid), dim3(B),
                           0, s, p, gas);
}

template <typename R>
void launch_dt_reduce(const DevPtrs<R>& p, hipStream_t s) {
    hipLaunchKernelGGL(k_dt_reduce, dim3(p.ninst), dim3(1024), 0, s, p.dt, (const double*)p.dt_part, p.finst_off,
                       p.tctl);
}

int residual_blocks(int nc) { return std::max(1, (nc + 255) / 256); }

template <typename R>
void launch_residual_norm(const DevPtrs<R>& p, double* out, hipStream_t s) {
    const int nb = residual_blocks(p.nc);
    hipLaunchKernelGGL(k_residual_part<R>, dim3(nb), dim3(256), 0, s, p);
    hipLaunchKernelGGL(k_residual_sum, dim3(1), dim3(1024), 0, s, (const double*)p.res_part, nb, out);
}

template <typename R>
void launch_flux_dt(const DevPtrs<R>& dev, double Rg, double Cv, double CFL, hipStream_t s) {
    unsigned grid;
    const DevPtrs<R> p = mapped(dev, flux_tiles(dev.nf, dev.nb), grid);
    const GasArgs gas = gas_args<R>(Rg, Cv, CFL);
    if (p.ngp > 0)
        hipLaunchKernelGGL((k_flux<R, true, true>), dim3(grid), dim3(256), 0, s, p, gas);
    else
        hipLaunchKernelGGL((k_flux<R, true, false>), dim3(grid), dim3(256), 0, s, p, gas);
}

template <typename R>
void launch_update(const DevPtrs<R>& p, double Rg, double gamma, double dt, const double* dt_ptr, double b1,
                   double b2, double b3, int last, hipStream_t s) {
    unsigned grid;
    const int B = small_blocks(p.nc) ? 64 : 256;
    const DevPtrs<R> q = mapped(p, std::max(1, (p.nc + B - 1) / B), grid);
    hipLaunchKernelGGL((B == 64 ? k_update<R, 64> : k_update<R, 256>), dim3(grid), dim3(B), 0, s, q, Rg, gamma, dt,
                       dt_ptr, b1, b2, b3, last);
}

template <typename R>
hipError_t set_lds_limits(size_t lds) {
    hipError_t e = hipSuccess;
#define AFAR_Q_KERNELS(GP, MS)                                                                     \
    (const void*)k_reconstruct_q<R, 64, GP, MS>, (const void*)k_reconstruct_q<R, 128, GP, MS>, \
        (const void*)k_reconstruct_q<R, 256, GP, MS>
    const void* fns[] = {(const void*)k_reconstruct<R, 64, false>,  (const void*)k_reconstruct<R, 128, false>,
                         (const void*)k_reconstruct<R, 256, false>, (const void*)k_reconstruct<R, 64, true>,
                         (const void*)k_reconstruct<R, 128, true>,  (const void*)k_reconstruct<R, 256, true>,
                         AFAR_Q_KERNELS(false, 8),                  AFAR_Q_KERNELS(false, 16),
                         AFAR_Q_KERNELS(false, kMaxSten),           AFAR_Q_KERNELS(true, 8),
                         AFAR_Q_KERNELS(true, 16),                  AFAR_Q_KERNELS(true, kMaxSten)};
#undef AFAR_Q_KERNELS
    for (const void* fn : fns) {
        // the dynamic limit plus the kernel's static LDS may not exceed the block limit
        hipFuncAttributes attr;
        e = hipFuncGetAttributes(&attr, fn);
        if (e != hipSuccess) return e;
        const size_t dyn = lds > attr.sharedSizeBytes ? lds - attr.sharedSizeBytes : 0;
        e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn);
        if (e != hipSuccess) return e;
    }
    return e;
}

#define AFAR_INSTANTIATE(R)                                                                                        \
    template void launch_lsq<R>(const DevPtrs<R>&, hipStream_t);                                                  \
    template void launch_cfl<R>(const DevPtrs<R>&, double, double, double, double*, hipStream_t);                          \
    template void launch_reconstruct<R>(const DevPtrs<R>&, int, size_t, hipStream_t, int);                        \
    template void launch_bvd<R>(const DevPtrs<R>&, int, size_t, hipStream_t);                                     \
    template void launch_flux<R>(const DevPtrs<R>&, double, double, hipStream_t);                                 \
    template void launch_flux_dt<R>(const DevPtrs<R>&, double, double, double, hipStream_t);                      \
    template void launch_dt_reduce<R>(const DevPtrs<R>&, hipStream_t);                                            \
    template void launch_residual_norm<R>(const DevPtrs<R>&, double*, hipStream_t);                               \
    template void launch_update<R>(const DevPtrs<R>&, double, double, double, const double*, double, double,      \
                                   double, int, hipStream_t);                                                     \
    template void launch_gather_fields<R>(const DevPtrs<R>&, const int32_t*, double4*, int8_t*, int, int,         \
                                          hipStream_t);                                                           \
    template hipError_t set_lds_limits<R>(size_t);

AFAR_INSTANTIATE(double)
AFAR_INSTANTIATE(float)

// Self-test entry: evaluates the shared elementary functions on the device.
__global__ void k_math_selftest(const double* x, double* out, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double v = x[i], w = x[n - 1 - i];
    double c[2], e[2];
    // as the flux calls them: two at once, x[i] the second (even i) or the first
    const bool first = i & 1;
    erfc_exp({first ? v : w, first ? w : v}, {first ? v : w, first ? w : v}, c, e);
    out[4 * i] = first ? e[0] : e[1];
    out[4 * i + 1] = first ? c[0] : c[1];
    out[4 * i + 2] = sqrt(v < 0 ? -v : v);
    out[4 * i + 3] = 1.0 / v;
}

__global__ void k_math_selftest_f32(const float* x, float* out, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = x[i], w = x[n - 1 - i];
    float c[2], e[2];
    const bool first = i & 1;
    erfc_exp({first ? v : w, first ? w : v}, {first ? v : w, first ? w : v}, c, e);
    out[4 * i] = first ? e[0] : e[1];
    out[4 * i + 1] = first ? c[0] : c[1];
    out[4 * i + 2] = sqrtf(v < 0 ? -v : v);
    out[4 * i + 3] = 1.0f / v;
}

void launch_math_selftest(const double* x, double* out, int n, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_math_selftest, dim3((n + 255) / 256), dim3(256), 0, s, x, out, n);
}

void launch_math_selftest_f32(const float* x, float* out, int n, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_math_selftest_f32, dim3((n + 255) / 256), dim3(256), 0, s, x, out, n);
}

}  // namespace afar
