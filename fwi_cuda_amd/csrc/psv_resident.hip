// psv_resident.hip -- the resident propagation (psv_resident.h): forward kernels, the tile
// choice and the receivers' running sums.
#include <algorithm>

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

// The tiling that takes the least time for nb shots on cus compute units with lds bytes each,
// by a model of a launch's step in us: its barriers and latencies, the two edge exchanges,
// the cells of a thread (a chain) and of the block (issue), the edge values.  Every tile
// holds at least N rows and columns (its halo comes from direct neighbours only).
bool plan_tiles(int nz, int nx, int N, int nb, int elt, int fields, int max_cpt, int cus, size_t lds,
                const std::vector<int> &zmap, const std::vector<int> &xmap, ResPlan *out) {
    const int iz = nz - 2 * N, ix = nx - 2 * N;
    double best = 1e300;
    const double e = elt / 4.0;
    for (int g = 1; g <= std::min(nb, cus); ++g) {
        const int launches = (nb + g - 1) / g, tiles = cus / g;
        if (g > 1 && (nb + g - 2) / (g - 1) == launches) continue;   // fewer shots a launch, as many launches
        for (int ntx = 1; ntx <= std::min(tiles, ix); ++ntx) {
            const int TX = (ix + ntx - 1) / ntx;
            if (TX > 64 || (ntx > 1 && ix - (ntx - 1) * TX < N)) continue;
            const int cols = strip_lines(xmap, N, TX);
            for (int ntz = 1; ntz <= std::min(tiles / ntx, iz); ++ntz)
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
                    const bool alone = ntx * ntz == 1;
                    double t = 1.0 + (alone ? 0.0 : 2.2) + 0.2 * cpt * e + 1.6e-3 * e * TX * TZ + 0.25e-3 * e * items;
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
    return best < 1e299;
}

}  // namespace

void launch_seis_scan(double *z, double *x, int rows, int nt, double dt, double dzdx, hipStream_t st) {
    if (rows > 0) hipLaunchKernelGGL(k_seis_scan, dim3(rows, 2), dim3(64), 0, st, z, x, nt, dt, dzdx);
}

// Cooperative launches work: the attribute, and one empty launch (the runtime's cooperative
// queue can be taken by another process of the same GPU; the steps then go launch by launch).
bool cooperative_ok(int device, hipStream_t st) {
    int a = 0;
    if (hipDeviceGetAttribute(&a, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess || !a) return false;
    if (hipLaunchCooperativeKernel((const void *)k_probe, dim3(1), dim3(64), nullptr, 0, st) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return true;
}

bool plan_resident(int nz, int nx, int N, int nb, int elt, int cus, size_t lds, const std::vector<int> &zmap,
                   const std::vector<int> &xmap, ResPlan *out) {
    return plan_tiles(nz, nx, N, nb, elt, 5, elt == 8 ? 4 : 8, cus, lds, zmap, xmap, out);
}

size_t resident_words(const ResPlan &p, int N, int elt) {
    return (size_t)2 * p.shots * p.ntx * p.ntz * 4 * N * (p.TX + p.TZ) * (elt / 4);
}

hipError_t launch_resident_forward(const ResArgs<float> &r, const ResPlan &p, int N, int shots, hipStream_t st) {
    return launch_resident_t<float, false>(r, N, p.cpt, shots * p.ntx * p.ntz, p.threads, p.lds, st);
}

}  // namespace psv
