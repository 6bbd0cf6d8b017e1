// psv_resident.h -- the resident propagation: a range of time steps in one launch.
//
// On small and middle-sized grids the two-kernel step is bound by its launches: four
// dependent kernels per time step (stress, velocity, sources, receivers) take 16 to 18 us
// whatever the grid, against 1 to 3 us of memory traffic.  Here one cooperative launch
// advances every step: a block per CU owns a tile of the interior and keeps its five
// fields, with a halo of N cells, in LDS, its media, energy and displacement in registers.
// Per half-step a block publishes its tile's edges and reads its neighbours'; nothing else
// leaves the chip but snapshots and receiver samples.  A step is then bound by the two edge
// exchanges (about 1.3 us each: a store to memory and a load from it, across the XCDs)
// and, from some 1000 cells per CU on, by the cells a thread computes.  Measured per time step
// of a call, launch by launch and resident: forward 72 x 96, 3 shots 16.4 -> 3.1 us, 201 x 401
// 17.7 -> 3.4 (both by k_resident1 below); the FP64 propagation at 201 x 401 beside the FP32 one
// 37 -> 8.9; a gradient (forward and adjoint) 201 x 401 37.5 -> 7.0, 246 x 335 order 4, 3 shots
// 36.6 -> 11.1, 301 x 601, 8 shots 90 -> 50.5 (two launches of four shots).
//
// Exchange.  An edge value travels as one 64-bit word {value, tag} (two for FP64, each
// half with its tag), stored and loaded with relaxed agent-scope atomics, so that one
// store and one load replace data, fence, flag and fence again.  The tag is a counter that
// never repeats within a context: a reader spins until the word carries the half-step it
// waits for.  One buffer per half-step is enough: a block overwrites its velocity words of
// step n in step n + 1, after it has seen its neighbours' stress words of step n + 1,
// which they write after the barrier that follows their reads of the velocity words (and
// likewise for the stress words).  Every wait ends: the launch is cooperative (all blocks
// are resident together), and a reader gives up after kSpinLimit loads, raises *err and
// waits no more.
//
// Work split.  A thread owns CPT cells of one column: the z taps of its CPT rows are
// CPT + 2N - 1 LDS reads per field instead of 2N CPT, the x taps are reads at constant
// offsets from neighbouring lanes' columns (no bank conflicts).  The arithmetic is that of
// stencil variant 5, in its order, and every product that is fused into a sum is written so
// (left to the compiler, a sum of two products fuses the one or the other as a tiling's
// unrolling has it): results do not depend on the tiling.
#pragma once

#include "psv_device.h"

#pragma clang fp contract(off)

namespace psv {
namespace {

__device__ __forceinline__ float fmadd(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmadd(double a, double b, double c) { return __builtin_fma(a, b, c); }

constexpr int kSpinLimit = 1 << 22;

template <class T>
__device__ __forceinline__ void mail_put(unsigned long long *w, T v, uint32_t tag) {
    if constexpr (sizeof(T) == 4) {
        __hip_atomic_store(w, (unsigned long long)__float_as_uint(v) | (unsigned long long)tag << 32, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    } else {
        const unsigned long long b = (unsigned long long)__double_as_longlong(v);
        __hip_atomic_store(w, (b & 0xffffffffull) | (unsigned long long)tag << 32, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(w + 1, (b >> 32) | (unsigned long long)tag << 32, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
}

__device__ __forceinline__ unsigned long long mail_get(const unsigned long long *w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// workgroup barrier that orders LDS only: edge words, samples and snapshots stay in flight
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The launch's arguments read again from the kernel-argument segment: inside the step loop
// through an opaque pointer, so that no argument and no address made from one is held in
// registers across the loop (held, they overflow the scalar registers and spill).
template <class R>
using RSegOf = const __attribute__((address_space(4))) R *;
template <class R>
__device__ __forceinline__ RSegOf<R> res_seg_of() {
    RSegOf<R> p = (RSegOf<R>)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}
template <class T>
using RSeg = RSegOf<ResArgs<T>>;
template <class T>
__device__ __forceinline__ RSeg<T> res_seg() {
    return res_seg_of<ResArgs<T>>();
}

// A tile's edges: the words it writes, and the words and LDS cells this thread reads.  A
// half-step exchanges two values per edge cell: LDS fields fr, fr + 1 across the rows'
// edges and fc, fc + 1 across the columns'.  LDS rows hold W values, A of each field.
template <class T, int N, int A, int W>
struct ResEdges {
    static constexpr int WPV = (int)sizeof(T) / 4;   // words per value
    int blk, ntx, TX, TZ, w, h, ev, eh;              // ev, eh: values of a rows' / columns' edge
    bool up, dn, lf, rt, dead;
    uint32_t tw, ph;                                 // words of a tile; of a half-step
    uint32_t mw[kResItems];
    int ml[kResItems];                               // LDS cell, + A for the second value; side in bits 28, 29
    int nit;

    __device__ __forceinline__ void init(int t, int nthr, int blk_, int ntx_, int ntz, int tx, int ty, int TX_, int TZ_,
                                         int w_, int h_, int blocks) {
        blk = blk_, ntx = ntx_, TX = TX_, TZ = TZ_, w = w_, h = h_;
        ev = 2 * N * TX, eh = 2 * N * TZ;
        tw = (uint32_t)(2 * ev + 2 * eh) * WPV;
        ph = tw * blocks;                            // the second half-step's words follow the first's
        up = ty > 0, dn = ty + 1 < ntz, lf = tx > 0, rt = tx + 1 < ntx;
        dead = false;
        nit = 0;
        const int nt_ = up ? 2 * N * w : 0, nb_ = dn ? 2 * N * w : 0, nl_ = lf ? 2 * N * h : 0, nr_ = rt ? 2 * N * h : 0;
#pragma unroll
        for (int q = 0; q < kResItems; ++q) {
            mw[q] = 0;
            ml[q] = 0;
            int i = t + q * nthr;
            if (i >= nt_ + nb_ + nl_ + nr_) continue;
            nit = q + 1;
            if (i < nt_ + nb_) {                     // rows: [value][row][column]
                const bool top = i < nt_;
                if (!top) i -= nt_;
                const int f = i / (N * w), row = i / w % N, col = i % w;
                const int tile = top ? blk - ntx : blk + ntx;
                mw[q] = tile * tw + (uint32_t)((top ? ev : 0) + (f * N + row) * TX + col) * WPV;
                ml[q] = ((top ? row : N + h + row) * W + N + col + f * A) | (top ? 0 : 1) << 28;
            } else {                                 // columns: [value][row][column]
                i -= nt_ + nb_;
                const bool left = i < nl_;
                if (!left) i -= nl_;
                const int f = i / (N * h), row = i / N % h, col = i % N;
                const int tile = left ? blk - 1 : blk + 1;
                mw[q] = tile * tw + (uint32_t)(2 * ev + (left ? eh : 0) + (f * TZ + row) * N + col) * WPV;
                ml[q] = ((N + row) * W + (left ? col : N + w + col) + f * A) | (left ? 2 : 3) << 28;
            }
        }
    }
    __device__ __forceinline__ int cell(int q, int fr, int fc) const {
        return (ml[q] & ((1 << 28) - 1)) + (ml[q] >> 29 & 1 ? fc : fr) * A;
    }
    // wait for the neighbours' words of a half-step and put them into the halo
    __device__ __forceinline__ void receive(T *lds, const unsigned long long *base, uint32_t tag, int fr, int fc, int *err) {
        unsigned long long v[kResItems][WPV];
#pragma unroll
        for (int q = 0; q < kResItems; ++q)
            if (q < nit)
#pragma unroll
                for (int j = 0; j < WPV; ++j) v[q][j] = mail_get(base + mw[q] + j);
#pragma unroll
        for (int q = 0; q < kResItems; ++q)
            if (q < nit) {
#pragma unroll
                for (int j = 0; j < WPV; ++j) {
                    int spin = 0;
                    while ((uint32_t)(v[q][j] >> 32) != tag && !dead) {
                        v[q][j] = mail_get(base + mw[q] + j);
                        if (++spin > kSpinLimit) {
                            dead = true;
                            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                        }
                    }
                }
                T val;
                if constexpr (sizeof(T) == 4)
                    val = __uint_as_float((uint32_t)v[q][0]);
                else
                    val = __longlong_as_double((long long)((v[q][0] & 0xffffffffull) | v[q][WPV - 1] << 32));
                lds[cell(q, fr, fc)] = val;
            }
    }
    // Publishing.  Threads of few cells write the words of their own cells (row z, column xc;
    // a, b go to the rows' edges, c, d to the columns').  With more cells a thread that does so
    // stalls its wavefront on a few lanes' stores per row, so after a barrier the threads
    // write the words that face the ones they read, in full runs.
    __device__ __forceinline__ void publish(unsigned long long *mail, uint32_t tag, int z, int xc, T a, T b, T c, T d) const {
        const bool eu = up && z < N, ed = dn && z >= h - N && z < h, el = lf && xc < N && z < h,
                   er = rt && xc >= w - N && z < h;
        if (!(eu || ed || el || er)) return;
        unsigned long long *o = mail + blk * tw;
        auto put = [&](uint32_t off, uint32_t second, T v1, T v2) {
            mail_put(o + off * WPV, v1, tag);
            mail_put(o + (off + second) * WPV, v2, tag);
        };
        if (eu) put((uint32_t)(z * TX + xc), (uint32_t)(N * TX), a, b);
        if (ed) put((uint32_t)(ev + (z - h + N) * TX + xc), (uint32_t)(N * TX), a, b);
        if (el) put((uint32_t)(2 * ev + z * N + xc), (uint32_t)(N * TZ), c, d);
        if (er) put((uint32_t)(2 * ev + eh + z * N + xc - w + N), (uint32_t)(N * TZ), c, d);
    }
    __device__ __forceinline__ void publish_runs(const T *lds, unsigned long long *mail, uint32_t tag, int fr, int fc) const {
#pragma unroll
        for (int q = 0; q < kResItems; ++q)
            if (q < nit) {
                const int e = ml[q] >> 28 & 3;       // 0 up, 1 down, 2 left, 3 right
                const int dw = e == 0 ? ntx * (int)tw - ev * WPV : e == 1 ? ev * WPV - ntx * (int)tw
                             : e == 2 ? (int)tw - eh * WPV : eh * WPV - (int)tw;
                const int dc = e == 0 ? N * W : e == 1 ? -N * W : e == 2 ? N : -N;
                mail_put(mail + (uint32_t)((int)mw[q] + dw), lds[cell(q, fr, fc) + dc], tag);
            }
    }
};

// profile k (b, a, 1/K at the integer point, then at the half point) of a grid line
__device__ __forceinline__ float prof_at(const ResArgs<float> &, const CpmlPoint &p, const float *, int, int k) {
    return k == 0 ? p.b : k == 1 ? p.a : k == 2 ? p.ik : k == 3 ? p.bh : k == 4 ? p.ah : p.ikh;
}
__device__ __forceinline__ double prof_at(const ResArgs<double> &, const CpmlPoint &, const double *pf, int i, int k) {
    return pf[(size_t)i * 6 + k];
}

template <class T, int N, int CPT, int LX, bool ADJ>
__global__ __launch_bounds__(1024) void k_resident(const ResArgs<T> r) {
    extern __shared__ char smem[];
    constexpr bool kReg = CPT <= 2;             // gradient sums in registers
    constexpr bool kOwn = CPT <= 4;             // edges published by their owners
    // CPML memory: in registers where they hold it, else in LDS (r.psi_lds) or the arrays
    constexpr bool kPsiReg = CPT * (int)sizeof(T) * (ADJ ? 2 : 1) <= 8;
    constexpr int QL = CPT + 2 * N - 1;         // rows a thread's z taps span
    const int t = threadIdx.x, nthr = blockDim.x;
    // LDS: [row][field][column], so that one register addresses every tap of a thread
    constexpr int A = LX + 2 * N, W = 5 * A;    // field and row stride
    const int TX = r.TX, TZ = r.TZ, rows = TZ + 2 * N;
    T *lvz = reinterpret_cast<T *>(smem), *lvx = lvz + A, *lzz = lvx + A, *lzx = lzz + A, *lxx = lzx + A;
    T *zprof = lvz + rows * W;                               // [TZ][6]
    int *zmapl = reinterpret_cast<int *>(zprof + TZ * 6);    // [TZ]
    T *lpsi = reinterpret_cast<T *>(zmapl + (TZ + 1) / 2 * 2);   // [4][psi_rows][TX], [4][TZ][psi_cols]

    const int blk = blockIdx.x, tx = blk % r.ntx, ty = blk / r.ntx % r.ntz, ls = blk / (r.ntx * r.ntz);
    const int s = r.s0 + ls;                    // shot of the batch
    const int x0 = N + tx * TX, z0 = N + ty * TZ;
    const int w = min(TX, r.nx - N - x0), h = min(TZ, r.nz - N - z0);
    const int x = t % LX, zc = t / LX * CPT;    // the thread's column and first row in the tile
    const int nc = x < w ? min(max(h - zc, 0), CPT) : 0;   // its cells
    // Threads with a column compute all their CPT rows: rows past the tile have media 0, so
    // their fields stay what they are (0, outside the grid).
    const bool act = x < w && zc < TZ;
    const bool top_row = act && z0 + zc == r.surf;
    const int ix = x0 + min(x, w - 1);
    const size_t P = r.P, fo = (size_t)s * r.fs;
    const T dt = r.dt;

    // ---- sources and receivers of the thread's cells: group + 1 in the low / high half
    int *cellmap = reinterpret_cast<int *>(smem);
    for (int i = t; i < TX * TZ; i += nthr) cellmap[i] = 0;
    __syncthreads();
    for (int k = 0; k < 2; ++k) {
        const SrcArgs &a = k ? r.rec : r.src;
        for (int g = t; g < a.ngroups; g += nthr) {
            const int cell = a.grp_cell[g], cz = cell / r.P - z0, cx = cell % r.P - x0;
            if (a.grp_shot[g] - r.shot0 == s && cz >= 0 && cz < h && cx >= 0 && cx < w)
                cellmap[cz * TX + cx] |= (g + 1) << (16 * k);
        }
        __syncthreads();
    }
    int pt[CPT];
    bool any_pt = false;
    int psrc = -1;                              // the first cell with a source
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        pt[k] = k < nc ? cellmap[(zc + k) * TX + x] : 0;
        any_pt = any_pt || pt[k];
        if (psrc < 0 && (pt[k] & 0xffff)) psrc = k;
    }
    __syncthreads();

    // ---- state with its halo (cells outside the interior are zero in the arrays)
    for (int j = t; j < rows * A; j += nthr) {
        const int iz = z0 - N + j / A, jx = x0 - N + j % A, i = j / A * W + j % A;
        const bool in = r.load && iz < r.nz && jx < r.nx;
        const size_t o = fo + (size_t)iz * P + jx;
        lvz[i] = in ? r.vz[o] : T(0);
        lvx[i] = in ? r.vx[o] : T(0);
        lzz[i] = in ? r.szz[o] : T(0);
        lzx[i] = in ? r.szx[o] : T(0);
        lxx[i] = in ? r.sxx[o] : T(0);
    }
    for (int i = t; i < TZ; i += nthr) {
        const int iz = z0 + min(i, h - 1);
        const CpmlPoint p = r.zp[iz];
        zmapl[i] = p.map;
        for (int k = 0; k < 6; ++k) zprof[i * 6 + k] = prof_at(r, p, r.zpf, iz, k);
    }
    const CpmlPoint xpt = r.xp[ix];
    const int xm = xpt.map;
    const T xb = prof_at(r, xpt, r.xpf, ix, 0), xa = prof_at(r, xpt, r.xpf, ix, 1), xk = prof_at(r, xpt, r.xpf, ix, 2),
            xbh = prof_at(r, xpt, r.xpf, ix, 3), xah = prof_at(r, xpt, r.xpf, ix, 4),
            xkh = prof_at(r, xpt, r.xpf, ix, 5);
    T lam[CPT], mu[CPT], muzx[CPT], rhoz[CPT], rhox[CPT], we[CPT], uz[CPT], ux[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        lam[k] = mu[k] = muzx[k] = rhoz[k] = rhox[k] = we[k] = uz[k] = ux[k] = T(0);
        if (k < nc) {
            const size_t m = (size_t)(z0 + zc + k) * P + ix;
            lam[k] = r.lam[m];
            mu[k] = r.mu[m];
            muzx[k] = r.muzx[m];
            rhoz[k] = r.rhoz[m];
            rhox[k] = r.rhox[m];
            if (r.energy) we[k] = r.We[fo + m];
            if constexpr (ADJ) {
                uz[k] = r.uz[fo + m];
                ux[k] = r.ux[fo + m];
            }
        }
    }
    __syncthreads();
    // CPML memory: slots 0..3 the z strips', 4..7 the x strips'
    auto psi_at = [&](RSeg<T> q, int j, int k, int z) -> T * {
        return j < 4 ? q->psi[j] + (size_t)s * q->nzs * q->P + (uint32_t)(zmapl[z + k] * q->P + ix)
                     : q->psi[j] + ((size_t)s * q->nz + z0) * q->nxs + (uint32_t)((z + k) * q->nxs + xm);
    };
    unsigned zin = 0;                           // rows inside a z strip, and inside an x strip
    const unsigned xin = xm >= 0 ? (1u << nc) - 1u : 0u;
#pragma unroll
    for (int k = 0; k < CPT; ++k)
        if (k < nc && zmapl[zc + k] >= 0) zin |= 1u << k;
    // strip rows and columns of the tile are consecutive: their first ones
    int zm0 = 0;
    for (int k = h - 1; k >= 0; --k)
        if (zmapl[k] >= 0) zm0 = zmapl[k];
    int xm0 = 0;
    for (int k = w - 1; k >= 0; --k) {
        const int m = r.xp[x0 + k].map;
        if (m >= 0) xm0 = m;
    }
    T pr[kPsiReg ? 8 : 1][CPT];
    auto psi_in = [&](int j, int k) { return ((j < 4 ? zin : xin) >> k & 1) != 0; };
    auto psi_l = [&](int j, int k, int z, int xc) -> T * {
        return lpsi + (j < 4 ? (j * r.psi_rows + zmapl[z + k] - zm0) * TX + xc
                             : 4 * r.psi_rows * TX + ((j - 4) * TZ + z + k) * r.psi_cols + xm - xm0);
    };
#pragma unroll
    for (int k = 0; k < CPT; ++k)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if constexpr (kPsiReg) {
                pr[j][k] = r.load && psi_in(j, k) ? *psi_at(res_seg<T>(), j, k, zc) : T(0);
            } else {
                if (r.psi_lds && psi_in(j, k)) *psi_l(j, k, zc, x) = r.load ? *psi_at(res_seg<T>(), j, k, zc) : T(0);
            }
        }
    // p1, p2 of a pass in one direction: the memories of slots j, j + 1 advanced
    auto memory = [&](int j, int k, int z, int xc, T b1, T a1, T d1, T b2, T a2, T d2, T &p1, T &p2) {
        auto advance = [&](T *m1, T *m2) {
            p1 = j < 4 ? fmadd(b1, *m1, a1 * d1) : fmadd(a1, d1, b1 * *m1);
            p2 = j < 4 ? fmadd(b2, *m2, a2 * d2) : fmadd(a2, d2, b2 * *m2);
            *m1 = p1;
            *m2 = p2;
        };
        if constexpr (kPsiReg) {
            advance(&pr[j][k], &pr[j + 1][k]);
        } else if (r.psi_lds) {
            advance(psi_l(j, k, z, xc), psi_l(j + 1, k, z, xc));
        } else {
            const RSeg<T> q = res_seg<T>();
            advance(psi_at(q, j, k, z), psi_at(q, j + 1, k, z));
        }
    };

    // ---- the snapshot lattice
    const bool lcol = ix >= r.snap_x1 && ix <= r.snap_x2 && (ix - r.snap_x1) % r.snap_dx == 0;
    unsigned lat = 0;                           // rows on it
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        const int iz = z0 + zc + k;
        if (k < nc && lcol && iz >= r.snap_z1 && iz <= r.snap_z2 && (iz - r.snap_z1) % r.snap_dz == 0) lat |= 1u << k;
    }
    auto lat_cell = [&](int z) {                // cell in a slab of row z of the tile
        return (z0 + z - r.snap_z1) / r.snap_dz * r.snx + (ix - r.snap_x1) / r.snap_dx;
    };
    const size_t slab = (size_t)r.snz * r.snx;
    const int ng = ADJ ? (r.gform ? 5 : 3) : 0;
    T gs[ADJ && kReg ? 5 : 1][CPT];
    if constexpr (ADJ && kReg) {
#pragma unroll
        for (int k = 0; k < CPT; ++k)
#pragma unroll
            for (int j = 0; j < 5; ++j) gs[j][k] = j < ng && (lat >> k & 1) ? r.g[j][(size_t)s * slab + lat_cell(zc + k)] : T(0);
    }

    ResEdges<T, N, A, W> ed;
    ed.init(t, nthr, blk, r.ntx, r.ntz, tx, ty, TX, TZ, w, h, gridDim.x);
    auto receive = [&](bool stress, uint32_t tag) {
        const RSeg<T> q = res_seg<T>();
        ed.receive(lvz, q->mail + (stress ? ed.ph : 0), tag, stress ? 2 : 0, stress ? 3 : 0, q->err);
    };
    auto publish_runs = [&](bool stress, uint32_t tag) {
        ed.publish_runs(lvz, res_seg<T>()->mail + (stress ? ed.ph : 0), tag, stress ? 2 : 0, stress ? 3 : 0);
    };

    // one source of a group: its two velocity increments (vsrc2)
    auto source_row = [&](int j, int it, int k, T &dz, T &dx) {
        const RSeg<T> q = res_seg<T>();
        const auto &a = q->src;
        const size_t row = (size_t)a.grp_idx[j] * a.nt + it;
        const double sc = a.scale_shot ? a.scale_shot[q->shot0 + s] : 1.0;
        const double fz = a.stf_z[row] * sc, fx = a.stf_x[row] * sc;
        if (a.type == 0) {
            dz = (T)(a.dt * (double)rhoz[k] * fz / a.dzdx);
            dx = (T)(a.dt * (double)rhox[k] * fx / a.dzdx);
        } else {
            dz = (T)fz;
            dx = (T)fx;
        }
    };

    for (int n = 0; n < r.nsteps; ++n) {
        const int it = r.t0 + r.dir * n;
        const uint32_t tag = r.epoch + (uint32_t)n;
        // the thread's row and column, opaque per step: no address is carried over the loop
        int zv = zc, xv = x;
        asm volatile("" : "+v"(zv), "+v"(xv));
        const int base = (zv + N) * W + xv + N;   // LDS cell of the thread's first row
        // the first source's increments, read ahead of the waits
        T pdz = T(0), pdx = T(0);
        if (psrc >= 0) {
#pragma unroll
            for (int k = 0; k < CPT; ++k)
                if (k == psrc) source_row(res_seg<T>()->src.grp_off[(pt[k] & 0xffff) - 1], it, k, pdz, pdx);
        }
        if (n > 0) receive(false, tag - 1u);
        lds_barrier();
        // ---- stress half-step
        if (act) {
            T qz[QL], qx[QL];                   // vz rows -N .., vx rows -N + 1 ..
#pragma unroll
            for (int j = 0; j < QL; ++j) {
                qz[j] = lvz[base + (j - N) * W];
                qx[j] = lvx[base + (j - N + 1) * W];
            }
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                const int c = base + k * W;
                T vz_z = 0, vx_z = 0, vz_x = 0, vx_x = 0;
#pragma unroll
                for (int i = 1; i <= N; ++i) {
                    vz_z = fmadd(r.cz[i - 1], qz[k + N + i - 1] - qz[k + N - i], vz_z);
                    vx_z = fmadd(r.cz[i - 1], qx[k + N + i - 1] - qx[k + N - i], vx_z);
                    vz_x = fmadd(r.cx[i - 1], lvz[c + i] - lvz[c + 1 - i], vz_x);
                    vx_x = fmadd(r.cx[i - 1], lvx[c + i - 1] - lvx[c - i], vx_x);
                }
                if (zin >> k & 1) {
                    const T *pf = zprof + (zv + k) * 6;
                    T p1, p2;
                    memory(0, k, zv, xv, pf[0], pf[1], vz_z, pf[3], pf[4], vx_z, p1, p2);
                    vz_z = fmadd(vz_z, pf[2], p1);
                    vx_z = fmadd(vx_z, pf[5], p2);
                }
                if (xin >> k & 1) {
                    T p1, p2;
                    memory(4, k, zv, xv, xb, xa, vx_x, xbh, xah, vz_x, p1, p2);
                    vx_x = fmadd(vx_x, xk, p1);
                    vz_x = fmadd(vz_x, xkh, p2);
                }
                if constexpr (!ADJ && sizeof(T) == 4) {   // the strain rates the reverse sweep reads
                    if (r.hist && k < nc) {
                        T *hp = res_seg<T>()->hist + ((size_t)(it - r.hist_base) * r.hist_B + s) * 5 * r.fs +
                                (uint32_t)((z0 + zv + k) * r.P + ix);
                        hp[0] = vz_z;
                        hp[r.fs] = vx_x;
                        hp[2 * r.fs] = vz_x + vx_z;
                    }
                }
                const T l = lam[k], m = mu[k];
                const T div = l * (vx_x + vz_z);
                T nzz = fmadd(dt, fmadd(T(2) * m, vz_z, div), lzz[c]);
                T nzx = fmadd(dt * muzx[k], vz_x + vx_z, lzx[c]);
                T nxx = fmadd(dt, fmadd(T(2) * m, vx_x, div), lxx[c]);
                if (k == 0 && top_row) {   // surf_mirror at row N (src/cpu/n_kernel_lib_PSV.cpp:297-301)
                    nzz = 0;
                    nzx = 0;
                    nxx = T(4) * dt * vx_x * fmadd(l, m, m * m) / fmadd(T(2), m, l);
                }
                lzz[c] = nzz;
                lzx[c] = nzx;
                lxx[c] = nxx;
                if constexpr (CPT > 2) __builtin_amdgcn_sched_barrier(0);
                if constexpr (kOwn) ed.publish(res_seg<T>()->mail + ed.ph, tag, zv + k, xv, nzz, nzx, nzx, nxx);
            }
        }
        if constexpr (!kOwn) {
            lds_barrier();
            publish_runs(true, tag);
        }
        // what a correlating step reads, ahead of the wait
        const bool gstep = ADJ && it % r.snap_dt == 0;
        T sn[ADJ && kReg ? 5 : 1][CPT];
        const size_t snoff = ADJ ? (size_t)s * r.sn_stride + (size_t)((it - r.tb) / r.snap_dt) * slab : 0;
        if constexpr (ADJ && kReg) {
            if (gstep && lat) {
                const RSeg<T> q = res_seg<T>();
#pragma unroll
                for (int k = 0; k < CPT; ++k) {
                    const size_t o = snoff + lat_cell(zv + k);
#pragma unroll
                    for (int j = 0; j < 5; ++j) sn[j][k] = lat >> k & 1 ? q->sn[j][o] : T(0);
                }
            }
        }
        receive(true, tag);
        lds_barrier();
        // ---- velocity half-step
        if (act) {
            T qzz[QL], qzx[QL];                 // szz rows -N + 1 .., szx rows -N ..
#pragma unroll
            for (int j = 0; j < QL; ++j) {
                qzz[j] = lzz[base + (j - N + 1) * W];
                qzx[j] = lzx[base + (j - N) * W];
            }
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                const int c = base + k * W;
                T szz_z = 0, szx_z = 0, szx_x = 0, sxx_x = 0;
#pragma unroll
                for (int i = 1; i <= N; ++i) {
                    szz_z = fmadd(r.cz[i - 1], qzz[k + N + i - 1] - qzz[k + N - i], szz_z);
                    szx_z = fmadd(r.cz[i - 1], qzx[k + N + i - 1] - qzx[k + N - i], szx_z);
                    szx_x = fmadd(r.cx[i - 1], lzx[c + i - 1] - lzx[c - i], szx_x);
                    sxx_x = fmadd(r.cx[i - 1], lxx[c + i] - lxx[c + 1 - i], sxx_x);
                }
                // the reference's slot mapping (src/cpu/n_kernel_PSV.cpp:142-146)
                if (zin >> k & 1) {
                    const T *pf = zprof + (zv + k) * 6;
                    T p1, p2;
                    memory(2, k, zv, xv, pf[0], pf[1], szz_z, pf[3], pf[4], szx_z, p1, p2);
                    szz_z = fmadd(szz_z, pf[2], p1);
                    szx_z = fmadd(szx_z, pf[5], p2);
                }
                if (xin >> k & 1) {
                    T p1, p2;
                    memory(6, k, zv, xv, xb, xa, sxx_x, xbh, xah, szx_x, p1, p2);
                    sxx_x = fmadd(sxx_x, xk, p1);
                    szx_x = fmadd(szx_x, xkh, p2);
                }
                if constexpr (!ADJ && sizeof(T) == 4) {   // the stress divergences
                    if (r.hist && k < nc) {
                        T *hp = res_seg<T>()->hist + (((size_t)(it - r.hist_base) * r.hist_B + s) * 5 + 3) * r.fs +
                                (uint32_t)((z0 + zv + k) * r.P + ix);
                        hp[0] = szx_x + szz_z;
                        hp[r.fs] = sxx_x + szx_z;
                    }
                }
                const T vz0 = lvz[c], vx0 = lvx[c];
                const T vz1 = fmadd(dt * rhoz[k], szx_x + szz_z, vz0);
                const T vx1 = fmadd(dt * rhox[k], sxx_x + szx_z, vx0);
                if constexpr (ADJ) {
                    uz[k] = fmadd(dt, vz0, uz[k]);
                    ux[k] = fmadd(dt, vx0, ux[k]);
                }
                if (r.energy) we[k] = we[k] + fmadd(vx1, vx1, vz1 * vz1);
                lvz[c] = vz1;
                lvx[c] = vx1;
                if constexpr (CPT > 2) __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (ADJ) {
            if (gstep && lat) {                 // fwi_grad2 (:439-484)
                const RSeg<T> q = res_seg<T>();
                // a thread of many cells reads all its slab cells and sums first: one latency
                T S[5][CPT], gm[kReg ? 1 : 5][CPT];
                int lc[CPT];
#pragma unroll
                for (int k = 0; k < CPT; ++k) {
                    lc[k] = lat >> k & 1 ? lat_cell(zv + k) : 0;
#pragma unroll
                    for (int j = 0; j < 5; ++j) {
                        if constexpr (kReg) {
                            S[j][k] = sn[j][k];
                        } else {
                            S[j][k] = q->sn[j][snoff + lc[k]];
                            gm[j][k] = j < ng ? q->g[j][(size_t)s * slab + lc[k]] : T(0);
                        }
                    }
                }
#pragma unroll
                for (int k = 0; k < CPT; ++k) {
                    if (!(lat >> k & 1)) continue;
                    const int c = base + k * W;
                    const T Vz = S[0][k], Vx = S[1][k], Szz = S[2][k], Szx = S[3][k], Sxx = S[4][k];
                    const T c_zz = lzz[c], c_xx = lxx[c], c_zx = lzx[c];
                    const T lm = lam[k] + mu[k];
                    const T il = r.gain_lm / (lm * lm), im = r.gain_lm / (mu[k] * mu[k]);
                    const T s1 = T(0.25) * il * (Szz + Sxx) * (c_zz + c_xx);
                    const T b2 = T(0.25) * im * (Szz - Sxx), d2 = c_zz - c_xx, b3 = Szx * c_zx;
                    auto add = [&](int j, T v) {
                        if constexpr (kReg) gs[j][k] = fmadd(r.gw, v, gs[j][k]);
                        else q->g[j][(size_t)s * slab + lc[k]] = fmadd(r.gw, v, gm[j][k]);
                    };
                    add(0, s1);
                    if (!r.gform) {
                        add(1, fmadd(b2, d2, fmadd(im, b3, s1)));
                        add(2, fmadd(uz[k], Vz, ux[k] * Vx));
                    } else {
                        add(1, s1 + b2 * d2);
                        add(2, dt * (lvz[c] * Vz));
                        add(3, im * b3);
                        add(4, dt * (lvx[c] * Vx));
                    }
                }
            }
        }
        if (any_pt) {
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                if (!pt[k]) continue;
                const int c = base + k * W;
                const int gsrc = (pt[k] & 0xffff) - 1, grec = (int)((unsigned)pt[k] >> 16) - 1;
                const RSeg<T> q = res_seg<T>();
                T vz1 = lvz[c], vx1 = lvx[c];
                if (gsrc >= 0) {                // vsrc2: the group's sources in source order
                    int j = q->src.grp_off[gsrc];
                    const int j1 = q->src.grp_off[gsrc + 1];
                    if (k == psrc) {
                        vz1 += pdz;
                        vx1 += pdx;
                        ++j;
                    }
                    for (; j < j1; ++j) {
                        T dz, dx;
                        source_row(j, it, k, dz, dx);
                        vz1 += dz;
                        vx1 += dx;
                    }
                    lvz[c] = vz1;
                    lvx[c] = vx1;
                }
                if (grec >= 0)                  // the velocity sample; k_seis_scan makes urec2's running sum
                    for (int j = q->rec.grp_off[grec]; j < q->rec.grp_off[grec + 1]; ++j) {
                        const size_t o = (size_t)q->rec.grp_idx[j] * q->rec.nt + it;
                        q->seis_z[o] = (double)vz1;
                        q->seis_x[o] = (double)vx1;
                    }
            }
        }
        if (n + 1 < r.nsteps) {
            if constexpr (kOwn) {
                if (act)
#pragma unroll
                    for (int k = 0; k < CPT; ++k) {
                        const T vz1 = lvz[base + k * W], vx1 = lvx[base + k * W];
                        ed.publish(res_seg<T>()->mail, tag, zv + k, xv, vz1, vx1, vz1, vx1);
                    }
            } else {
                lds_barrier();
                publish_runs(false, tag);
            }
        }
        if constexpr (!ADJ) {
            if (r.store && lat && it >= r.tb && it % r.snap_dt == 0) {   // gard_fwd_storage2, after the injection
                const RSeg<T> q = res_seg<T>();
                const size_t so = (size_t)s * q->st_stride + (size_t)((it - q->tb) / q->snap_dt) * slab;
#pragma unroll
                for (int k = 0; k < CPT; ++k) {
                    if (!(lat >> k & 1)) continue;
                    const size_t o = so + lat_cell(zv + k);
                    const int c = base + k * W;
                    q->st[0][o] = lvz[c] / dt;
                    q->st[1][o] = lvx[c] / dt;
                    q->st[2][o] = lzz[c];
                    q->st[3][o] = lzx[c];
                    q->st[4][o] = lxx[c];
                }
            }
        }
        if constexpr (ADJ) {
            if ((r.nt - it) % r.flush_every == 0 && lat) {   // the FP32 sums into their FP64 totals
                const RSeg<T> q = res_seg<T>();
#pragma unroll
                for (int k = 0; k < CPT; ++k) {
                    if (!(lat >> k & 1)) continue;
                    const size_t o = (size_t)s * slab + lat_cell(zv + k);
#pragma unroll
                    for (int j = 0; j < 5; ++j) {
                        if (j >= ng) continue;
                        if constexpr (kReg) {
                            q->g64[j * q->g64_stride + o] += (double)gs[j][k];
                            gs[j][k] = T(0);
                        } else {
                            q->g64[j * q->g64_stride + o] += (double)q->g[j][o];
                            q->g[j][o] = T(0);
                        }
                    }
                }
            }
        }
    }

    // ---- the state back
    if (!r.load) return;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        if (k >= nc) continue;
        const size_t o = fo + (size_t)(z0 + zc + k) * P + ix;
        const int c = (zc + k + N) * W + x + N;
        r.vz[o] = lvz[c];
        r.vx[o] = lvx[c];
        r.szz[o] = lzz[c];
        r.szx[o] = lzx[c];
        r.sxx[o] = lxx[c];
        if (r.energy) r.We[o] = we[k];
        if constexpr (ADJ) {
            r.uz[o] = uz[k];
            r.ux[o] = ux[k];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (!psi_in(j, k)) continue;
            if constexpr (kPsiReg) {
                *psi_at(res_seg<T>(), j, k, zc) = pr[j][k];
            } else {
                if (r.psi_lds) *psi_at(res_seg<T>(), j, k, zc) = *psi_l(j, k, zc, x);
            }
        }
        if constexpr (ADJ && kReg) {
#pragma unroll
            for (int j = 0; j < 5; ++j)
                if (j < ng && (lat >> k & 1)) r.g[j][(size_t)s * slab + lat_cell(zc + k)] = gs[j][k];
        }
    }
}

// One exchange per step, for small tiles.  A thread owns one cell of the tile or of the N
// cells around it and advances the stresses there too (the same operations on the same
// values as their owner, so the same bits); only velocities travel, 2N cells deep.  A step
// then waits once instead of twice, for N more rows and columns of stress arithmetic each
// side and more words: worth it where a CU has threads to spare (at most 32 - 2N rows and
// 31 - 2N columns per tile).  A tile's words are its own lines of memory, two sets taken in turn: a block
// overwrites the words of step n in step n + 2, after it has seen every neighbour's words
// of step n + 1, which they write after the barrier that follows their reads of step n.
// The rim is loaded from arrays that its owners overwrite when they end: a block stores its
// state only after it has seen a word of every neighbour, which they write after their
// loads.  From two steps on the exchange sees to that; a launch of one step makes the
// exchange for that alone (k_resident waits for stress words in every step, and the exact
// adjoint's sweep loads own cells only).
// Measured per time step of a call, two exchanges and one: 72 x 96, 3 shots 4.2 -> 3.1 us, 201 x
// 401 3.8 -> 3.4; forward and adjoint 201 x 401 8.1 -> 7.0.  The FP64 propagation's words are
// twice as many: with one exchange its step took a tenth longer, so it keeps two.  A tile's
// words lie together: at their cell's place in one array (lines written by several blocks) a
// step of 17 x 15 tiles took an eighth longer; rows of 32 lanes: packed to the tile's width
// they take fewer wavefronts, and a step 8 % longer.
template <int N, bool ADJ>
__global__ __launch_bounds__(1024) void k_resident1(const ResArgs<float> r) {
    extern __shared__ char smem[];
    using T = float;
    constexpr int VA = 32 + 2 * N, VW = 2 * VA, SA = 32, SW = 3 * SA;
    const int t = threadIdx.x, nthr = blockDim.x;
    const int TX = r.TX, TZ = r.TZ;
    T *lvz = reinterpret_cast<T *>(smem), *lvx = lvz + VA;                 // [TZ + 4N][2][VA]
    T *lzz = lvz + (TZ + 4 * N) * VW, *lzx = lzz + SA, *lxx = lzx + SA;    // [TZ + 2N][3][SA]
    T *zprof = lzz + (TZ + 2 * N) * SW;                                    // [TZ + 2N][6]
    const int blk = blockIdx.x, tx = blk % r.ntx, ty = blk / r.ntx % r.ntz, ls = blk / (r.ntx * r.ntz);
    const int s = r.s0 + ls;
    const int x0 = N + tx * TX, z0 = N + ty * TZ;
    const int w = min(TX, r.nx - N - x0), h = min(TZ, r.nz - N - z0);
    const int lx = t % 32, lz = t / 32;                    // cell (x0 - N + lx, z0 - N + lz)
    const int ix = x0 - N + lx, iz = z0 - N + lz;
    const bool own = lx >= N && lx < N + w && lz >= N && lz < N + h;
    const bool ext = lx < w + 2 * N && lz < h + 2 * N && ix >= N && ix < r.nx - N && iz >= N && iz < r.nz - N;
    const size_t P = r.P, fo = (size_t)s * r.fs;
    const size_t m = ext ? (size_t)iz * P + ix : 0;
    const T dt = r.dt;

    int *cellmap = reinterpret_cast<int *>(smem);
    for (int i = t; i < 32 * (TZ + 2 * N); i += nthr) cellmap[i] = 0;
    __syncthreads();
    for (int k = 0; k < 2; ++k) {
        const SrcArgs &a = k ? r.rec : r.src;
        for (int g = t; g < a.ngroups; g += nthr) {
            const int cell = a.grp_cell[g], cz = cell / r.P - z0, cx = cell % r.P - x0;
            if (a.grp_shot[g] - r.shot0 == s && cz >= 0 && cz < h && cx >= 0 && cx < w)
                cellmap[(cz + N) * 32 + cx + N] |= (g + 1) << (16 * k);
        }
        __syncthreads();
    }
    const int pt = own ? cellmap[lz * 32 + lx] : 0;
    const int gsrc = (pt & 0xffff) - 1, grec = (int)((unsigned)pt >> 16) - 1;
    __syncthreads();

    for (int j = t; j < (TZ + 4 * N) * VA; j += nthr) {
        const int cz = z0 - 2 * N + j / VA, cx = x0 - 2 * N + j % VA, i = j / VA * VW + j % VA;
        const bool in = r.load && cz >= 0 && cz < r.nz && cx >= 0 && cx < r.nx;
        const size_t o = fo + (size_t)cz * P + cx;
        lvz[i] = in ? r.vz[o] : T(0);
        lvx[i] = in ? r.vx[o] : T(0);
    }
    for (int j = t; j < (TZ + 2 * N) * SW; j += nthr) lzz[j] = T(0);
    for (int i = t; i < TZ + 2 * N; i += nthr) {
        const int cz = min(max(z0 - N + i, 0), r.nz - 1);
        const CpmlPoint p = r.zp[cz];
        for (int k = 0; k < 6; ++k) zprof[i * 6 + k] = prof_at(r, p, r.zpf, cz, k);
    }
    const CpmlPoint xpt = r.xp[ext ? ix : N];
    const int cxp = ext ? ix : N;
    const int xm = ext ? xpt.map : -1, zm = ext ? r.zp[iz].map : -1;
    const T xb = prof_at(r, xpt, r.xpf, cxp, 0), xa = prof_at(r, xpt, r.xpf, cxp, 1), xk = prof_at(r, xpt, r.xpf, cxp, 2),
            xbh = prof_at(r, xpt, r.xpf, cxp, 3), xah = prof_at(r, xpt, r.xpf, cxp, 4),
            xkh = prof_at(r, xpt, r.xpf, cxp, 5);
    const T lam = ext ? r.lam[m] : T(0), mu = ext ? r.mu[m] : T(0), muzx = ext ? r.muzx[m] : T(0);
    const T rhoz = own ? r.rhoz[m] : T(0), rhox = own ? r.rhox[m] : T(0);
    const bool ld = r.load && ext;
    T szz = ld ? r.szz[fo + m] : T(0), szx = ld ? r.szx[fo + m] : T(0), sxx = ld ? r.sxx[fo + m] : T(0);
    T vz = ld && own ? r.vz[fo + m] : T(0), vx = ld && own ? r.vx[fo + m] : T(0);
    T we = own && r.energy ? r.We[fo + m] : T(0), uz = T(0), ux = T(0);
    if constexpr (ADJ) {
        if (own) uz = r.uz[fo + m], ux = r.ux[fo + m];
    }
    auto psi_at = [&](RSeg<T> q, int j) -> T * {
        return j < 4 ? q->psi[j] + ((size_t)s * q->nzs + zm) * q->P + ix
                     : q->psi[j] + ((size_t)s * q->nz + iz) * q->nxs + xm;
    };
    // the stress pass's memories (slots 0, 1, 4, 5) belong to every cell the thread advances,
    // the velocity pass's to its own
    auto psi_in = [&](int j) { return (j < 4 ? zm >= 0 : xm >= 0) && ((j & 2) == 0 || own); };
    T pr[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) pr[j] = r.load && psi_in(j) ? *psi_at(res_seg<T>(), j) : T(0);
    const bool zs = zm >= 0, xs = xm >= 0, top_row = ext && iz == r.surf;

    const bool lat = own && ix >= r.snap_x1 && ix <= r.snap_x2 && (ix - r.snap_x1) % r.snap_dx == 0 &&
                     iz >= r.snap_z1 && iz <= r.snap_z2 && (iz - r.snap_z1) % r.snap_dz == 0;
    const uint32_t lc = lat ? (uint32_t)((iz - r.snap_z1) / r.snap_dz * r.snx + (ix - r.snap_x1) / r.snap_dx) : 0u;
    const size_t slab = (size_t)r.snz * r.snx;
    const int ng = ADJ ? (r.gform ? 5 : 3) : 0;
    T gs[ADJ ? 5 : 1];
    if constexpr (ADJ) {
#pragma unroll
        for (int j = 0; j < 5; ++j) gs[j] = j < ng && lat ? r.g[j][(size_t)s * slab + lc] : T(0);
    }

    // the words this thread reads: velocities of the cells within 2N of the tile
    const uint32_t tw = res1_words(TX, TZ), set = gridDim.x * tw;   // words of a tile, of a set
    auto word = [&](int cz, int cx) {           // of the cell's owner
        const int ox = (cx - N) / TX, oz = (cz - N) / TZ;
        return (uint32_t)((ls * r.ntz + oz) * r.ntx + ox) * tw +
               (uint32_t)((cz - N - oz * TZ) * TX + cx - N - ox * TX) * 2u;
    };
    uint32_t mw[kRes1Cells];
    int ml[kRes1Cells];
    int nit = 0;
#pragma unroll
    for (int q = 0; q < kRes1Cells; ++q) {
        mw[q] = 0;
        ml[q] = -1;
        const int i = t + q * nthr;
        if (i >= (w + 4 * N) * (h + 4 * N)) continue;
        const int rx = i % (w + 4 * N), rz = i / (w + 4 * N), cx = x0 - 2 * N + rx, cz = z0 - 2 * N + rz;
        if (cx < N || cx >= r.nx - N || cz < N || cz >= r.nz - N) continue;
        if (rx >= 2 * N && rx < 2 * N + w && rz >= 2 * N && rz < 2 * N + h) continue;
        mw[q] = word(cz, cx);
        ml[q] = rz * VW + rx;
        nit = q + 1;
    }
    const uint32_t mine = own ? word(iz, ix) : 0u;
    bool dead = false;
    auto receive = [&](uint32_t tag, int parity) {
        const RSeg<T> sg = res_seg<T>();
        const unsigned long long *base = sg->mail + (parity ? set : 0u);
        unsigned long long v[kRes1Cells][2];
#pragma unroll
        for (int q = 0; q < kRes1Cells; ++q)
            if (ml[q] >= 0)
#pragma unroll
                for (int j = 0; j < 2; ++j) v[q][j] = mail_get(base + mw[q] + j);
#pragma unroll
        for (int q = 0; q < kRes1Cells; ++q)
            if (ml[q] >= 0) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    int spin = 0;
                    while ((uint32_t)(v[q][j] >> 32) != tag && !dead) {
                        v[q][j] = mail_get(base + mw[q] + j);
                        if (++spin > kSpinLimit) {
                            dead = true;
                            __hip_atomic_store(sg->err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                        }
                    }
                }
#pragma unroll
                for (int f = 0; f < 2; ++f) lvz[ml[q] + f * VA] = __uint_as_float((uint32_t)v[q][f]);
            }
    };
    auto source_row = [&](int j, int it, T &dz, T &dx) {
        const RSeg<T> q = res_seg<T>();
        const auto &a = q->src;
        const size_t row = (size_t)a.grp_idx[j] * a.nt + it;
        const double sc = a.scale_shot ? a.scale_shot[q->shot0 + s] : 1.0;
        const double fz = a.stf_z[row] * sc, fx = a.stf_x[row] * sc;
        if (a.type == 0) {
            dz = (T)(a.dt * (double)rhoz * fz / a.dzdx);
            dx = (T)(a.dt * (double)rhox * fx / a.dzdx);
        } else {
            dz = (T)fz;
            dx = (T)fx;
        }
    };
    __syncthreads();

    const int vc = (lz + N) * VW + lx + N, sc_ = lz * SW + lx;   // the cell in the two LDS planes
    for (int n = 0; n < r.nsteps; ++n) {
        const int it = r.t0 + r.dir * n;
        const uint32_t tag = r.epoch + (uint32_t)n;
        int c = vc, d = sc_;
        asm volatile("" : "+v"(c), "+v"(d));
        T pdz = T(0), pdx = T(0);               // the first source's increments, read ahead of the wait
        if (gsrc >= 0) source_row(res_seg<T>()->src.grp_off[gsrc], it, pdz, pdx);
        const bool gstep = ADJ && it % r.snap_dt == 0;
        T S[ADJ ? 5 : 1];
        if constexpr (ADJ) {
            if (gstep && lat) {                 // what a correlating step reads, too
                const RSeg<T> q = res_seg<T>();
                const size_t o = (size_t)s * q->sn_stride + (size_t)((it - q->tb) / q->snap_dt) * slab + lc;
#pragma unroll
                for (int j = 0; j < 5; ++j) S[j] = q->sn[j][o];
            }
        }
        if (n > 0 && nit) receive(tag - 1u, (n - 1) & 1);
        lds_barrier();
        if (ext) {                              // ---- stress half-step
            T vz_z = 0, vx_z = 0, vz_x = 0, vx_x = 0;
#pragma unroll
            for (int i = 1; i <= N; ++i) {
                vz_z = fmadd(r.cz[i - 1], lvz[c + (i - 1) * VW] - lvz[c - i * VW], vz_z);
                vx_z = fmadd(r.cz[i - 1], lvx[c + i * VW] - lvx[c - (i - 1) * VW], vx_z);
                vz_x = fmadd(r.cx[i - 1], lvz[c + i] - lvz[c + 1 - i], vz_x);
                vx_x = fmadd(r.cx[i - 1], lvx[c + i - 1] - lvx[c - i], vx_x);
            }
            if (zs) {
                const T *pf = zprof + lz * 6;
                const T p1 = fmadd(pf[0], pr[0], pf[1] * vz_z), p2 = fmadd(pf[3], pr[1], pf[4] * vx_z);
                pr[0] = p1;
                pr[1] = p2;
                vz_z = fmadd(vz_z, pf[2], p1);
                vx_z = fmadd(vx_z, pf[5], p2);
            }
            if (xs) {
                const T p1 = fmadd(xa, vx_x, xb * pr[4]), p2 = fmadd(xah, vz_x, xbh * pr[5]);
                pr[4] = p1;
                pr[5] = p2;
                vx_x = fmadd(vx_x, xk, p1);
                vz_x = fmadd(vz_x, xkh, p2);
            }
            if constexpr (!ADJ) {
                if (r.hist && own) {
                    T *hp = res_seg<T>()->hist + ((size_t)(it - r.hist_base) * r.hist_B + s) * 5 * r.fs + m;
                    hp[0] = vz_z;
                    hp[r.fs] = vx_x;
                    hp[2 * r.fs] = vz_x + vx_z;
                }
            }
            const T div = lam * (vx_x + vz_z);
            szz = fmadd(dt, fmadd(T(2) * mu, vz_z, div), szz);
            szx = fmadd(dt * muzx, vz_x + vx_z, szx);
            sxx = fmadd(dt, fmadd(T(2) * mu, vx_x, div), sxx);
            if (top_row) {                      // surf_mirror at row N (src/cpu/n_kernel_lib_PSV.cpp:297-301)
                szz = 0;
                szx = 0;
                sxx = T(4) * dt * vx_x * fmadd(lam, mu, mu * mu) / fmadd(T(2), mu, lam);
            }
            lzz[d] = szz;
            lzx[d] = szx;
            lxx[d] = sxx;
        }
        lds_barrier();
        if (own) {                              // ---- velocity half-step
            T szz_z = 0, szx_z = 0, szx_x = 0, sxx_x = 0;
#pragma unroll
            for (int i = 1; i <= N; ++i) {
                szz_z = fmadd(r.cz[i - 1], lzz[d + i * SW] - lzz[d - (i - 1) * SW], szz_z);
                szx_z = fmadd(r.cz[i - 1], lzx[d + (i - 1) * SW] - lzx[d - i * SW], szx_z);
                szx_x = fmadd(r.cx[i - 1], lzx[d + i - 1] - lzx[d - i], szx_x);
                sxx_x = fmadd(r.cx[i - 1], lxx[d + i] - lxx[d + 1 - i], sxx_x);
            }
            if (zs) {
                const T *pf = zprof + lz * 6;
                const T p1 = fmadd(pf[0], pr[2], pf[1] * szz_z), p2 = fmadd(pf[3], pr[3], pf[4] * szx_z);
                pr[2] = p1;
                pr[3] = p2;
                szz_z = fmadd(szz_z, pf[2], p1);
                szx_z = fmadd(szx_z, pf[5], p2);
            }
            if (xs) {
                const T p1 = fmadd(xa, sxx_x, xb * pr[6]), p2 = fmadd(xah, szx_x, xbh * pr[7]);
                pr[6] = p1;
                pr[7] = p2;
                sxx_x = fmadd(sxx_x, xk, p1);
                szx_x = fmadd(szx_x, xkh, p2);
            }
            if constexpr (!ADJ) {
                if (r.hist) {
                    T *hp = res_seg<T>()->hist + (((size_t)(it - r.hist_base) * r.hist_B + s) * 5 + 3) * r.fs + m;
                    hp[0] = szx_x + szz_z;
                    hp[r.fs] = sxx_x + szx_z;
                }
            }
            const T vz0 = vz, vx0 = vx;
            T vz1 = fmadd(dt * rhoz, szx_x + szz_z, vz0);
            T vx1 = fmadd(dt * rhox, sxx_x + szx_z, vx0);
            if constexpr (ADJ) {
                uz = fmadd(dt, vz0, uz);
                ux = fmadd(dt, vx0, ux);
            }
            if (r.energy) we = we + fmadd(vx1, vx1, vz1 * vz1);
            const T pvz = vz1, pvx = vx1;       // before the injection
            if (gsrc >= 0) {                    // vsrc2: the group's sources in source order
                const RSeg<T> q = res_seg<T>();
                vz1 += pdz;
                vx1 += pdx;
                for (int j = q->src.grp_off[gsrc] + 1; j < q->src.grp_off[gsrc + 1]; ++j) {
                    T dz, dx;
                    source_row(j, it, dz, dx);
                    vz1 += dz;
                    vx1 += dx;
                }
            }
            vz = vz1;
            vx = vx1;
            lvz[c] = vz1;
            lvx[c] = vx1;
            if (n + 1 < r.nsteps || n == 0) {
                unsigned long long *o = res_seg<T>()->mail + (n & 1 ? set : 0u) + mine;
                mail_put(o, vz1, tag);
                mail_put(o + 1, vx1, tag);
            }
            if (grec >= 0) {                    // the velocity sample; k_seis_scan makes urec2's running sum
                const RSeg<T> q = res_seg<T>();
                for (int j = q->rec.grp_off[grec]; j < q->rec.grp_off[grec + 1]; ++j) {
                    const size_t o = (size_t)q->rec.grp_idx[j] * q->rec.nt + it;
                    q->seis_z[o] = (double)vz1;
                    q->seis_x[o] = (double)vx1;
                }
            }
            if constexpr (ADJ) {
                if (lat) {
                    if (gstep) {                // fwi_grad2 (:439-484)
                        const T Vz = S[0], Vx = S[1], Szz = S[2], Szx = S[3], Sxx = S[4];
                        const T lm = lam + mu;
                        const T il = r.gain_lm / (lm * lm), im = r.gain_lm / (mu * mu);
                        const T s1 = T(0.25) * il * (Szz + Sxx) * (szz + sxx);
                        const T b2 = T(0.25) * im * (Szz - Sxx), d2 = szz - sxx, b3 = Szx * szx;
                        gs[0] = fmadd(r.gw, s1, gs[0]);
                        if (!r.gform) {
                            gs[1] = fmadd(r.gw, fmadd(b2, d2, fmadd(im, b3, s1)), gs[1]);
                            gs[2] = fmadd(r.gw, fmadd(uz, Vz, ux * Vx), gs[2]);
                        } else {
                            gs[1] = fmadd(r.gw, s1 + b2 * d2, gs[1]);
                            gs[2] = fmadd(r.gw, dt * (pvz * Vz), gs[2]);
                            gs[3] = fmadd(r.gw, im * b3, gs[3]);
                            gs[4] = fmadd(r.gw, dt * (pvx * Vx), gs[4]);
                        }
                    }
                    if ((r.nt - it) % r.flush_every == 0) {   // the FP32 sums into their FP64 totals
                        const RSeg<T> q = res_seg<T>();
#pragma unroll
                        for (int j = 0; j < 5; ++j)
                            if (j < ng) {
                                q->g64[j * q->g64_stride + (size_t)s * slab + lc] += (double)gs[j];
                                gs[j] = T(0);
                            }
                    }
                }
            } else {
                if (r.store && lat && it >= r.tb && it % r.snap_dt == 0) {   // gard_fwd_storage2
                    const RSeg<T> q = res_seg<T>();
                    const size_t o = (size_t)s * q->st_stride + (size_t)((it - q->tb) / q->snap_dt) * slab + lc;
                    q->st[0][o] = vz1 / dt;
                    q->st[1][o] = vx1 / dt;
                    q->st[2][o] = szz;
                    q->st[3][o] = szx;
                    q->st[4][o] = sxx;
                }
            }
        }
    }

    if (r.nsteps == 1) {                        // the neighbours have loaded their rims
        if (nit) receive(r.epoch, 0);
        lds_barrier();
    }
    if (!r.load || !own) return;
    r.vz[fo + m] = vz;
    r.vx[fo + m] = vx;
    r.szz[fo + m] = szz;
    r.szx[fo + m] = szx;
    r.sxx[fo + m] = sxx;
    if (r.energy) r.We[fo + m] = we;
    if constexpr (ADJ) {
        r.uz[fo + m] = uz;
        r.ux[fo + m] = ux;
#pragma unroll
        for (int j = 0; j < 5; ++j)
            if (j < ng && lat) r.g[j][(size_t)s * slab + lc] = gs[j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
        if (psi_in(j)) *psi_at(res_seg<T>(), j) = pr[j];
}

template <class T, bool ADJ, int N>
hipError_t launch_resident_n(const ResArgs<T> &r, int cpt, int blocks, int threads, size_t lds, hipStream_t st) {
    constexpr int E = (int)sizeof(T);
    const void *f = cpt == 1   ? (const void *)k_resident<T, N, 1, res_lanes(1, E), ADJ>
                    : cpt == 2 ? (const void *)k_resident<T, N, 2, res_lanes(2, E), ADJ>
                               : (const void *)k_resident<T, N, 4, res_lanes(4, E), ADJ>;
    if constexpr (E == 4) {
        if (cpt == 0) f = (const void *)k_resident1<N, ADJ>;
        if (cpt == 8) f = (const void *)k_resident<T, N, 8, res_lanes(8, E), ADJ>;
    }
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    void *args[] = {const_cast<ResArgs<T> *>(&r)};
    return hipLaunchCooperativeKernel(f, dim3(blocks), dim3(threads), args, (unsigned)lds, st);
}

template <class T, bool ADJ>
hipError_t launch_resident_t(const ResArgs<T> &r, int N, int cpt, int blocks, int threads, size_t lds, hipStream_t st) {
    switch (N) {
        case 1: return launch_resident_n<T, ADJ, 1>(r, cpt, blocks, threads, lds, st);
        case 2: return launch_resident_n<T, ADJ, 2>(r, cpt, blocks, threads, lds, st);
        case 3: return launch_resident_n<T, ADJ, 3>(r, cpt, blocks, threads, lds, st);
        case 4: return launch_resident_n<T, ADJ, 4>(r, cpt, blocks, threads, lds, st);
        case 5: return launch_resident_n<T, ADJ, 5>(r, cpt, blocks, threads, lds, st);
        default: return launch_resident_n<T, ADJ, 6>(r, cpt, blocks, threads, lds, st);
    }
}

}  // namespace
}  // namespace psv
