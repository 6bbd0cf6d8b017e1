// psv_resident_exact.hip -- the exact adjoint's reverse sweep in one launch.
//
// psv_exact.hip's reverse step is eleven dependent launches (the receivers' adjoint
// sources, the two passes, their gathers, the surface and the clears between them), 45 us
// a step at 201 x 401 whose traffic takes 5.  Here a block per CU keeps its tile for the
// whole sweep as in psv_resident.h, with the same exchange: the adjoint state, the CPML
// carries and the FP64 media gradient stay in registers (carries of tall threads in LDS),
// and LDS holds the four derivative adjoints of one half-step, whose z and x gathers need
// the neighbours' edge rows and columns.  The step's history is read ahead of the waits.
// Bound by the exchanges and barriers: 6.0 us a step at 201 x 401; by issue beside them: 11.5
// per launch of two shots at 301 x 601.  A call with the forward pass before it: 201 x 401, 800
// steps 63.4 -> 11.4 ms; 301 x 601, 4 shots, 400 steps 66.4 -> 19.4 ms, with the workspace kept.
// Same operations in the same order as psv_exact.hip's kernels, with their fused products but
// for one (d3; over eight models of 201 x 401 its form here leaves lam, mu errors of 1.61,
// 2.01e-6 against 64 bits, theirs 1.66, 2.18e-6), for no free surface or the top one at row N
// (no image rows) and points inside the interior; other set-ups keep those kernels.
#include "psv_resident.h"

namespace psv {
namespace {

template <int N, int CPT, int LX>
__global__ __launch_bounds__(1024) void k_resident_exact(const ResExact r) {
    extern __shared__ char smem[];
    using Seg = RSegOf<ResExact>;
    constexpr bool kPsiReg = CPT <= 2;   // CPML carries in registers
    constexpr int QL = CPT + 2 * N - 1;
    constexpr int A = LX + 2 * N, W = 4 * A;
    const int t = threadIdx.x, nthr = blockDim.x;
    const int TX = r.TX, TZ = r.TZ, rows = TZ + 2 * N;
    float *l0 = reinterpret_cast<float *>(smem), *l1 = l0 + A, *l2 = l1 + A, *l3 = l2 + A;
    float *zprof = l0 + rows * W;
    int *zmapl = reinterpret_cast<int *>(zprof + TZ * 6);
    float *lpsi = reinterpret_cast<float *>(zmapl + (TZ + 1) / 2 * 2);
    const int blk = blockIdx.x, tx = blk % r.ntx, ty = blk / r.ntx % r.ntz, s = r.s0 + blk / (r.ntx * r.ntz);
    const int x0 = N + tx * TX, z0 = N + ty * TZ;
    const int w = min(TX, r.nx - N - x0), h = min(TZ, r.nz - N - z0);
    const int x = t % LX, zc = t / LX * CPT;
    const int nc = x < w ? min(max(h - zc, 0), CPT) : 0;
    const bool act = x < w && zc < TZ;
    const bool top_row = act && z0 + zc == r.surf;
    const int ix = x0 + min(x, w - 1);
    const size_t fo = (size_t)s * r.fs;
    const float dt = r.dt;

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
    int psrc = -1;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        pt[k] = k < nc ? cellmap[(zc + k) * TX + x] : 0;
        any_pt = any_pt || pt[k];
        if (psrc < 0 && (pt[k] & 0xffff)) psrc = k;
    }
    __syncthreads();
    for (int i = t; i < rows * W; i += nthr) l0[i] = 0.f;
    for (int i = t; i < TZ; i += nthr) {
        const CpmlPoint p = r.zp[z0 + min(i, h - 1)];
        zmapl[i] = p.map;
        const float v[6] = {p.b, p.a, p.ik, p.bh, p.ah, p.ikh};
        for (int k = 0; k < 6; ++k) zprof[i * 6 + k] = v[k];
    }
    const CpmlPoint xq = r.xp[ix];
    const int xm = xq.map;
    float lam[CPT], mu[CPT], muzx[CPT], rhoz[CPT], rhox[CPT], bvz[CPT], bvx[CPT], bzz[CPT], bzx[CPT], bxx[CPT];
    double G[5][CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        const bool in = k < nc;
        const size_t m = in ? (size_t)(z0 + zc + k) * r.P + ix : 0;
        lam[k] = in ? r.lam[m] : 0.f;
        mu[k] = in ? r.mu[m] : 0.f;
        muzx[k] = in ? r.muzx[m] : 0.f;
        rhoz[k] = in ? r.rhoz[m] : 0.f;
        rhox[k] = in ? r.rhox[m] : 0.f;
        bvz[k] = in ? r.bvz[fo + m] : 0.f;
        bvx[k] = in ? r.bvx[fo + m] : 0.f;
        bzz[k] = in ? r.bzz[fo + m] : 0.f;
        bzx[k] = in ? r.bzx[fo + m] : 0.f;
        bxx[k] = in ? r.bxx[fo + m] : 0.f;
        for (int j = 0; j < 5; ++j) G[j][k] = in ? r.G[((size_t)s * 5 + j) * r.fs + m] : 0.0;
    }
    __syncthreads();
    unsigned zin = 0;
    const unsigned xin = xm >= 0 ? (1u << nc) - 1u : 0u;
#pragma unroll
    for (int k = 0; k < CPT; ++k)
        if (k < nc && zmapl[zc + k] >= 0) zin |= 1u << k;
    int zm0 = 0, xm0 = 0;
    for (int k = h - 1; k >= 0; --k)
        if (zmapl[k] >= 0) zm0 = zmapl[k];
    for (int k = w - 1; k >= 0; --k) {
        const int m = r.xp[x0 + k].map;
        if (m >= 0) xm0 = m;
    }
    auto psi_at = [&](Seg q, int j, int k, int z) -> float * {
        return j < 4 ? q->psi[j] + (size_t)s * q->nzs * q->P + (uint32_t)(zmapl[z + k] * q->P + ix)
                     : q->psi[j] + ((size_t)s * q->nz + z0) * q->nxs + (uint32_t)((z + k) * q->nxs + xm);
    };
    auto psi_in = [&](int j, int k) { return ((j < 4 ? zin : xin) >> k & 1) != 0; };
    auto psi_l = [&](int j, int k, int z, int xc) -> float * {
        return lpsi + (j < 4 ? (j * r.psi_rows + zmapl[z + k] - zm0) * TX + xc
                             : 4 * r.psi_rows * TX + ((j - 4) * TZ + z + k) * r.psi_cols + xm - xm0);
    };
    float pr[kPsiReg ? 8 : 1][CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if constexpr (kPsiReg) {
                pr[j][k] = psi_in(j, k) ? *psi_at(res_seg_of<ResExact>(), j, k, zc) : 0.f;
            } else {
                if (r.psi_lds && psi_in(j, k)) *psi_l(j, k, zc, x) = *psi_at(res_seg_of<ResExact>(), j, k, zc);
            }
        }
    // the CPML recursion reversed on slots j (b1, a1, k1, d1) and j + 1: q = carry + d,
    // d = d / K + a q, carry = b q
    auto memory = [&](int j, int k, int z, int xc, float b1, float a1, float k1, float &d1, float b2, float a2, float k2,
                      float &d2) {
        auto advance = [&](float *m1, float *m2) {
            float q = *m1 + d1;
            d1 = fmadd(d1, k1, a1 * q);
            *m1 = b1 * q;
            q = *m2 + d2;
            d2 = fmadd(d2, k2, a2 * q);
            *m2 = b2 * q;
        };
        if constexpr (kPsiReg) {
            advance(&pr[j][k], &pr[j + 1][k]);
        } else if (r.psi_lds) {
            advance(psi_l(j, k, z, xc), psi_l(j + 1, k, z, xc));
        } else {
            const Seg q = res_seg_of<ResExact>();
            advance(psi_at(q, j, k, z), psi_at(q, j + 1, k, z));
        }
    };
    ResEdges<float, N, A, W> ed;
    ed.init(t, nthr, blk, r.ntx, r.ntz, tx, ty, TX, TZ, w, h, gridDim.x);

    for (int n = 0; n < r.nsteps; ++n) {
        const int it = r.t0 - n;
        const uint32_t tag = r.epoch + (uint32_t)n;
        int zv = zc, xv = x;
        asm volatile("" : "+v"(zv), "+v"(xv));
        const int base = (zv + N) * W + xv + N;
        // the step's history: e_zz e_xx e_zx S_z S_x
        float hs[5][CPT];
        {
            const float *hp = res_seg_of<ResExact>()->hist + ((size_t)(it - r.hist_base) * r.hist_B + s) * 5 * r.fs;
#pragma unroll
            for (int k = 0; k < CPT; ++k)
#pragma unroll
                for (int j = 0; j < 5; ++j)
                    hs[j][k] = k < nc ? hp[j * r.fs + (uint32_t)((z0 + zv + k) * r.P + ix)] : 0.f;
        }
        if (any_pt) {
            const Seg q = res_seg_of<ResExact>();
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                if (!pt[k]) continue;
                const int gsrc = (pt[k] & 0xffff) - 1, grec = (int)((unsigned)pt[k] >> 16) - 1;
                if (gsrc >= 0)       // v' += A (the running sum's transpose)
                    for (int j = q->src.grp_off[gsrc]; j < q->src.grp_off[gsrc + 1]; ++j) {
                        const size_t row = (size_t)q->src.grp_idx[j] * q->src.nt + it;
                        bvz[k] += (float)q->src.stf_z[row];
                        bvx[k] += (float)q->src.stf_x[row];
                    }
                if (grec >= 0) {     // type-0 sources: the inverse density in the injected amount
                    double fz = 0.0, fx = 0.0;
                    for (int j = q->rec.grp_off[grec]; j < q->rec.grp_off[grec + 1]; ++j) {
                        const size_t row = (size_t)q->rec.grp_idx[j] * q->rec.nt + it;
                        fz += q->rec.stf_z[row];
                        fx += q->rec.stf_x[row];
                    }
                    G[3][k] += (double)bvz[k] * q->rec.dt * fz / q->rec.dzdx;
                    G[4][k] += (double)bvx[k] * q->rec.dt * fx / q->rec.dzdx;
                }
            }
        }
        // ---- velocity update reversed: density terms, stress-derivative adjoints
        if (act) {
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                const int c = base + k * W;
                const float az = bvz[k], ax = bvx[k];
                G[3][k] = fmadd((double)az * dt, (double)hs[3][k], G[3][k]);
                G[4][k] = fmadd((double)ax * dt, (double)hs[4][k], G[4][k]);
                const float tz = dt * rhoz[k] * az, tx_ = dt * rhox[k] * ax;
                float d0 = tz, d2 = tz, d1 = tx_, d3 = tx_;   // szz_z, szx_x; szx_z, sxx_x
                if (zin >> k & 1) {
                    const float *p = zprof + (zv + k) * 6;
                    memory(2, k, zv, xv, p[0], p[1], p[2], d0, p[3], p[4], p[5], d1);
                }
                if (xin >> k & 1) memory(6, k, zv, xv, xq.b, xq.a, xq.ik, d3, xq.bh, xq.ah, xq.ikh, d2);
                l0[c] = d0;
                l1[c] = d1;
                l2[c] = d2;
                l3[c] = d3;
                ed.publish(res_seg_of<ResExact>()->mail, tag, zv + k, xv, d0, d1, d2, d3);
            }
        }
        {
            const Seg q = res_seg_of<ResExact>();
            ed.receive(l0, q->mail, tag, 0, 2, q->err);
        }
        lds_barrier();
        // ---- stress-derivative transposes gathered
        if (act) {
            float q0[QL], q1[QL];                   // D0 rows -N .., D1 rows -N + 1 ..
#pragma unroll
            for (int j = 0; j < QL; ++j) {
                q0[j] = l0[base + (j - N) * W];
                q1[j] = l1[base + (j - N + 1) * W];
            }
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                const int c = base + k * W;
                float zz = 0.f, zx = 0.f, xx = 0.f;
#pragma unroll
                for (int i = 1; i <= N; ++i) {
                    zz = fmadd(r.cz[i - 1], q0[k + N - i] - q0[k + N + i - 1], zz);
                    zx = fmadd(r.cz[i - 1], q1[k + N - i] - q1[k + N + i - 1], zx);
                    zx = fmadd(r.cx[i - 1], l2[c - i + 1] - l2[c + i], zx);
                    xx = fmadd(r.cx[i - 1], l3[c - i] - l3[c + i - 1], xx);
                }
                bzz[k] = k < nc ? bzz[k] + zz : 0.f;
                bzx[k] = k < nc ? bzx[k] + zx : 0.f;
                bxx[k] = k < nc ? bxx[k] + xx : 0.f;
            }
        }
        lds_barrier();
        // ---- free surface and stress update reversed: media gradient, strain-rate adjoints
        if (act) {
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                const int c = base + k * W;
                float s3 = 0.f;
                if (k == 0 && top_row) {
                    const double l = lam[0], u = mu[0], den = fmadd(2.0, u, l);
                    const double f = fmadd(l, u, u * u) / den, f_l = u * u / (den * den),
                                 f_u = fmadd(2.0 * u, u, fmadd(l, l, 2.0 * l * u)) / (den * den);
                    const double a = bxx[0], e = hs[1][0];
                    s3 = (float)(a * 4.0 * dt * f);
                    G[0][0] = fmadd(a * 4.0 * dt * e, f_l, G[0][0]);
                    G[1][0] = fmadd(a * 4.0 * dt * e, f_u, G[1][0]);
                    bzz[0] = bzx[0] = bxx[0] = 0.f;
                }
                const float zz = bzz[k], zx = bzx[k], xx = bxx[k];
                const float e_zz = hs[0][k], e_xx = hs[1][k], e_zx = hs[2][k], l = lam[k], u = mu[k];
                G[0][k] = fmadd((double)dt * ((double)zz + xx), (double)e_xx + e_zz, G[0][k]);
                G[1][k] = fmadd(2.0 * dt, fmadd((double)zz, (double)e_zz, (double)xx * e_xx), G[1][k]);
                G[2][k] = fmadd((double)dt * zx, (double)e_zx, G[2][k]);
                const float lu = fmadd(2.f, u, l);
                float d0 = dt * fmadd(l, xx, lu * zz);
                float d3 = fmadd(dt, fmadd(lu, xx, l * zz), s3);   // the larger product fused: as one cell per thread had it
                float d1 = dt * muzx[k] * zx, d2 = d1;
                if (zin >> k & 1) {
                    const float *p = zprof + (zv + k) * 6;
                    memory(0, k, zv, xv, p[0], p[1], p[2], d0, p[3], p[4], p[5], d1);
                }
                if (xin >> k & 1) memory(4, k, zv, xv, xq.b, xq.a, xq.ik, d3, xq.bh, xq.ah, xq.ikh, d2);
                l0[c] = d0;
                l1[c] = d1;
                l2[c] = d2;
                l3[c] = d3;
                ed.publish(res_seg_of<ResExact>()->mail + ed.ph, tag, zv + k, xv, d0, d1, d2, d3);
            }
        }
        {
            const Seg q = res_seg_of<ResExact>();
            ed.receive(l0, q->mail + ed.ph, tag, 0, 2, q->err);
        }
        lds_barrier();
        // ---- velocity-derivative transposes gathered
        if (act) {
            float q0[QL], q1[QL];                   // D0 rows -N + 1 .., D1 rows -N ..
#pragma unroll
            for (int j = 0; j < QL; ++j) {
                q0[j] = l0[base + (j - N + 1) * W];
                q1[j] = l1[base + (j - N) * W];
            }
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                const int c = base + k * W;
                float vz = 0.f, vx = 0.f;
#pragma unroll
                for (int i = 1; i <= N; ++i) {
                    vz = fmadd(r.cz[i - 1], q0[k + N - i] - q0[k + N + i - 1], vz);
                    vz = fmadd(r.cx[i - 1], l2[c - i] - l2[c + i - 1], vz);
                    vx = fmadd(r.cz[i - 1], q1[k + N - i] - q1[k + N + i - 1], vx);
                    vx = fmadd(r.cx[i - 1], l3[c - i + 1] - l3[c + i], vx);
                }
                bvz[k] = k < nc ? bvz[k] + vz : 0.f;
                bvx[k] = k < nc ? bvx[k] + vx : 0.f;
            }
        }
        lds_barrier();
    }

#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        if (k >= nc) continue;
        const size_t m = (size_t)(z0 + zc + k) * r.P + ix;
        r.bvz[fo + m] = bvz[k];
        r.bvx[fo + m] = bvx[k];
        r.bzz[fo + m] = bzz[k];
        r.bzx[fo + m] = bzx[k];
        r.bxx[fo + m] = bxx[k];
        for (int j = 0; j < 5; ++j) r.G[((size_t)s * 5 + j) * r.fs + m] = G[j][k];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (!psi_in(j, k)) continue;
            if constexpr (kPsiReg) {
                *psi_at(res_seg_of<ResExact>(), j, k, zc) = pr[j][k];
            } else {
                if (r.psi_lds) *psi_at(res_seg_of<ResExact>(), j, k, zc) = *psi_l(j, k, zc, x);
            }
        }
    }
}

template <int N>
hipError_t launch_n(const ResExact &r, const ResPlan &p, int blocks, hipStream_t st) {
    const void *f = p.cpt == 1   ? (const void *)k_resident_exact<N, 1, res_lanes(1, 4)>
                    : p.cpt == 2 ? (const void *)k_resident_exact<N, 2, res_lanes(2, 4)>
                                 : (const void *)k_resident_exact<N, 4, res_lanes(4, 4)>;
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds);
    if (e != hipSuccess) return e;
    void *args[] = {const_cast<ResExact *>(&r)};
    return hipLaunchCooperativeKernel(f, dim3(blocks), dim3(p.threads), args, (unsigned)p.lds, st);
}

}  // namespace

hipError_t launch_resident_exact(const ResExact &r, const ResPlan &p, int N, int shots, hipStream_t st) {
    const int blocks = shots * p.ntx * p.ntz;
    switch (N) {
        case 1: return launch_n<1>(r, p, blocks, st);
        case 2: return launch_n<2>(r, p, blocks, st);
        case 3: return launch_n<3>(r, p, blocks, st);
        case 4: return launch_n<4>(r, p, blocks, st);
        case 5: return launch_n<5>(r, p, blocks, st);
        default: return launch_n<6>(r, p, blocks, st);
    }
}

}  // namespace psv
