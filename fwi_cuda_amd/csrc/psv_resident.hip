// psv_resident.hip -- the resident propagation (psv_resident.h): forward kernels, the tile
// choice and the receivers' running sums.
#include <algorithm>
#include <atomic>

#include "psv_resident.h"

namespace psv {
namespace {

// urec2 (src/cpu/n_kernel_lib_PSV.cpp:538-576) on rows of velocity samples, in place: the
// running sum of dt v / (dz dx) in time order.  A wavefront per row: its lanes turn the
// next 64 samples into increments and lane 0's order is kept by adding them one by one,
// so the sums are those of k_record bit for bit; a row's samples move in 512-byte runs.
__global__ __launch_bounds__(64) void k_seis_scan(double *z, double *x, int nt, double dt, double dzdx) {
    double *p = (blockIdx.y ? x : z) + (size_t)blockIdx.x * nt;
    double acc = 0.0;
    for (int t0 = 0; t0 < nt; t0 += 64) {
        const int t = t0 + threadIdx.x;
        const double d = t < nt ? dt * p[t] / dzdx : 0.0;
        double mine = 0.0;
        for (int l = 0; l < 64; ++l) {
            acc += __shfl(d, l);
            if (l == (int)threadIdx.x) mine = acc;
        }
        if (t < nt) p[t] = mine;
    }
}

__global__ void k_probe() {}

size_t res_lds(int N, int elt, int fields, int cpt, int TZ) {
    return (size_t)fields * elt * (res_lanes(cpt, elt) + 2 * N) * (TZ + 2 * N) + (size_t)TZ * 6 * elt +
           (size_t)(TZ + 1) / 2 * 8;
}

// the most strip lines a tile of T interior lines holds
int strip_lines(const std::vector<int> &map, int N, int T) {
    const int end = (int)map.size() - N;
    int most = 0;
    for (int a = N; a < end; a += T) {
        int n = 0;
        for (int i = a; i < std::min(a + T, end); ++i) n += map[i] >= 0;
        most = std::max(most, n);
    }
    return most;
}

}  // namespace

// The tiling that takes the least time for nb shots on cus compute units with lds bytes each,
// by a model of step times in us: a base (the barriers and latencies of the chain of a thread's
// cells, and the two edge exchanges) and a slope per lane-cell of the block, fitted to sweeps of
// tiles (of use to compare them, not for a call's time).  Measured there with one cell per
// thread: 3.8 at 300 cells, 4.4 at 740; two: 5.6 at 450, 6.5 at 1600; four: 10.8 at 3300;
// eight (its registers spill): 25 at 4600.  FP64 and the exact adjoint's sweep cost what
// their registers and words do; that sweep with four cells per thread spills its FP64 sums
// (301 x 601, 4 shots: 31 us a step against 2 x 11.5 for two launches of two cells per
// thread).  Every tile holds at least N rows and columns, as its halo comes from direct
// neighbours only (the one-exchange kernel, 0 cells per thread, reads any tile's words).  FP32
// steps that the batched kernels run as fast, at 16 us of launches and 14.4 us per million
// cells, are left to them: 600 x 1100, 8 shots take 78 us there and 82 here, 800 x 1400, 1
// shot 35 and 26.
bool plan_resident(int nz, int nx, int N, int nb, ResUse use, int cus, size_t lds, const std::vector<int> &zmap,
                   const std::vector<int> &xmap, ResPlan *out) {
    const int elt = use == kUseFp64 ? 8 : 4, fields = use == kUseExact ? 4 : 5;
    const int max_cpt = use == kUseStep || use == kUseExactForward ? 8 : 4;
    const int iz = nz - 2 * N, ix = nx - 2 * N;
    double best = 1e300;
    const double e = use == kUseFp64 ? 1.8 : use == kUseExact ? 1.5 : 1.0;
    for (int g = 1; g <= std::min(nb, cus); ++g) {
        const int launches = (nb + g - 1) / g, tiles = cus / g;
        if (g > 1 && (nb + g - 2) / (g - 1) == launches) continue;   // fewer shots a launch, as many launches
        for (int ntx = 1; ntx <= std::min(tiles, ix); ++ntx) {
            const int TX = (ix + ntx - 1) / ntx;
            if (TX > 64 || (ntx > 1 && ix - (ntx - 1) * TX < N)) continue;
            const int cols = strip_lines(xmap, N, TX);
            for (int ntz = 1; ntz <= std::min(tiles / ntx, iz); ++ntz) {
                // one exchange per step (a single tile has none: one cell per thread); tiles that
                // fill the 32 lanes measured 5 % slower than narrower ones (201 x 401: 24 x 13
                // cells against 22 x 14 and 16 x 20, which take the same time)
                if (use != kUseExact && use != kUseFp64 && TX + 2 * N < 32 && ntx * ntz > 1) {
                    const int TZ = (iz + ntz - 1) / ntz;
                    const int thr = (32 * (TZ + 2 * N) + 63) / 64 * 64;
                    if (thr <= 1024 && iz - (ntz - 1) * TZ > 0 &&
                        (TX + 4 * N) * (TZ + 4 * N) <= kRes1Cells * thr) {
                        // tiles narrower than the frame (narrow grids, orders 10 and 12) wait for
                        // their neighbours' neighbours too
                        const bool thin = (ntx > 1 && TX < 2 * N) || (ntz > 1 && TZ < 2 * N);
                        const double t = launches * (2.3 + (thin ? 0.5 : 0.0) + 1.1e-3 * thr);
                        if (t < best) {
                            best = t;
                            *out = {g, TX, TZ, ntx, ntz, 0, thr, 0, 0, 0,
                                    (size_t)elt * (2 * (32 + 2 * N) * (TZ + 4 * N) + (3 * 32 + 6) * (TZ + 2 * N))};
                        }
                    }
                }
                for (int cpt : {1, 2, 4, 8}) {
                    if (cpt > max_cpt || TX > res_lanes(cpt, elt)) continue;
                    const int rows = (iz + ntz - 1) / ntz, TZ = (rows + cpt - 1) / cpt * cpt;
                    const int lastz = iz - (ntz - 1) * TZ;
                    if (lastz <= 0 || (ntz > 1 && lastz < N)) continue;
                    const int thr = (res_lanes(cpt, elt) * (TZ / cpt) + 63) / 64 * 64;
                    size_t need = res_lds(N, elt, fields, cpt, TZ);
                    if (thr > 1024 || need > lds) continue;
                    const int items = (ntz > 1 ? 4 * N * TX : 0) + (ntx > 1 ? 4 * N * TZ : 0);
                    if (items > kResItems * thr) continue;
                    const double base = cpt == 1 ? 3.5 : cpt == 2 ? 5.0 : cpt == 4 ? 5.2 : 7.0;
                    const double slope = cpt <= 2 ? 0.9e-3 : cpt == 4 ? (use == kUseExact ? 3e-3 : 1.75e-3) : 3.9e-3;
                    double t = base - (ntx * ntz == 1 ? 2.4 : 0.0) + e * slope * res_lanes(cpt, elt) * TZ +
                               e * 0.25e-3 * items;
                    const int srows = strip_lines(zmap, N, TZ);
                    const size_t psi = (size_t)4 * elt * (srows * TX + cols * TZ);
                    const bool psi_lds = need + psi <= lds;
                    if (psi_lds) need += psi;
                    else t += 0.8 * cpt;
                    if (t * launches < best) {
                        best = t * launches;
                        *out = {g, TX, TZ, ntx, ntz, cpt, thr, psi_lds, srows, cols, need};
                    }
                }
            }
        }
    }
    out->us = best;
    return best < (use == kUseStep ? 0.9 * (16.0 + 14.4e-6 * nb * nz * nx) : 1e299);
}

// Cooperative launches work: the attribute, and one empty launch (the runtime's cooperative
// queue can be taken by another process of the same GPU; the steps then go launch by launch).
// Once made, a process's queue stays, so a device that took the launch is not asked again.
bool cooperative_ok(int device, hipStream_t st) {
    static std::atomic<unsigned long long> known{0};
    const unsigned long long bit = 1ull << (device & 63);
    if (device < 64 && (known.load() & bit)) return true;
    int a = 0;
    if (hipDeviceGetAttribute(&a, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess || !a) return false;
    if (hipLaunchCooperativeKernel((const void *)k_probe, dim3(1), dim3(64), nullptr, 0, st) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (device < 64) known.fetch_or(bit);
    return true;
}

void launch_seis_scan(double *z, double *x, int rows, int nt, double dt, double dzdx, hipStream_t st) {
    if (rows > 0) hipLaunchKernelGGL(k_seis_scan, dim3(rows, 2), dim3(64), 0, st, z, x, nt, dt, dzdx);
}

size_t resident_words(const ResPlan &p, int N, int elt) {
    if (p.cpt == 0) return (size_t)2 * p.shots * p.ntx * p.ntz * res1_words(p.TX, p.TZ);
    return (size_t)2 * p.shots * p.ntx * p.ntz * 4 * N * (p.TX + p.TZ) * (elt / 4);
}

hipError_t launch_resident_forward(const ResArgs<float> &r, const ResPlan &p, int N, int shots, hipStream_t st) {
    return launch_resident_t<float, false>(r, N, p.cpt, shots * p.ntx * p.ntz, p.threads, p.lds, st);
}

}  // namespace psv
