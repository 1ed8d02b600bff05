// Imaging condition of the adjoint run (gfx950): nl_we_op_a / nl_we_op_e / nl_we_op_vti
// ::compute_gradients (we_op.cpp:1555-1605, 488-565, 1108-1216), FP64 accumulation. One
// launch per kept snapshot.
//
// What bounds it: HBM traffic. An elastic event reads 60 B per cell (the slot, the field the
// derivatives are taken of, the adjoint field and the two neighbouring slots, FP32 store) and
// reads and writes 48 B of FP64 gradients. Workgroups of 32 z x 16 x points (512 threads)
// march along y over a chunk of planes: the y neighbours of a point stay in registers, the x
// and z neighbours (2-cell halos, loaded one plane ahead by the first 192 threads) pass
// through two LDS planes with one barrier per plane, so that a field value is read once per
// tile. Per event: elastic 200^3 FP32 290 us (3.0 TB/s of those 108 B per cell), 256^3 BF16 488
// us, 131 x 141 x 153 FP16 120 us, VTI 150 x 144 x 71 87 us, acoustic 128^3 28 us. One
// workgroup per 64 x 4 tile and plane, its y neighbours read from memory, took 473, 848, 158,
// 131 and 35 us.
// Closure rows along x and z take a window of 6 points with weights, as in the fused step;
// along y they are whole planes and read memory.
#pragma once
#include "fused.hpp"

namespace fwi3d {

template <int NF>
struct ImagingSmem {
    float pad[8];                     // (a z window may start one point before the plane)
    float u[2][NF][FPX][FPZ];         // plane mod 2, field, x row (from x0-2), z column (from z0-2)
};

// Tiling of an event: ntz x ntx tiles, y chunks of `chunk` planes; workgroup b -> tile and
// chunk with z fastest, each XCD a contiguous range (halos meet in its L2).
struct ImagingTiles { int ntz, ntx, nyc, chunk; };
inline ImagingTiles imaging_tiles(const Geom& g) {
    ImagingTiles T;
    T.ntz = fused_tile_count(g.nz, FZ);
    T.ntx = fused_tile_count(g.nx, FW);
    // about 1024 workgroups (two rounds of two per CU), at least 4 planes each: a chunk
    // reads 4 planes of its own column ahead
    const int want = std::max(1, 1024 / (T.ntz * T.ntx));
    T.chunk = std::max(4, (g.ny + want - 1) / want);
    T.nyc = (g.ny + T.chunk - 1) / T.chunk;
    return T;
}

// March over one tile and chunk: NC components of the forward slot fn and of `lag`. Per plane
// begin(p, i) and, when the derivatives are formed, end(i, F, L, fv, lv), for points to output:
// p is the point's index in a field, i its index in the unpadded gradients, F and L the
// derivatives of the forward components and of lag, [axis x, y, z][component], fv and lv
// their values at the point.
template <int NC, int FMT, class Begin, class End>
__device__ __forceinline__ void imaging_march(ImagingSmem<2 * NC>& S, const SnapView<FMT>& fn, const float* __restrict__ lag,
                                              const Geom& g, const ImagingTiles& T, const Begin& begin, const End& end) {
    constexpr int CP = FPX * FPZ, PL = 2 * NC * CP;
    const int nx = g.nx, ny = g.ny, nz = g.nz, sx = g.sx, sy = g.sy, n3 = g.n;
    const int b = xcd_remap(blockIdx.x, T.ntz * T.ntx * T.nyc);
    const int tz = b % T.ntz, tx = (b / T.ntz) % T.ntx, ch = b / (T.ntz * T.ntx);
    const int ya = ch * T.chunk, yb = min(ny, ya + T.chunk);
    int z0, zo0, zo1, x0, xo0, xo1;
    fused_tile(nz, FZ, tz, T.ntz, z0, zo0, zo1);
    fused_tile(nx, FW, tx, T.ntx, x0, xo0, xo1);
    const bool XE = tx == 0 || tx == T.ntx - 1, ZE = tz == 0 || tz == T.ntz - 1;
    const int t = threadIdx.x, lz = t & (FZ - 1), lx = t >> 5;
    const int ix = x0 + lx, iz = z0 + lz;
    const int col = min(ix, nx - 1) * sx + min(iz, nz - 1);
    const bool outp = ix >= xo0 && ix < xo1 && iz >= zo0 && iz < zo1;
    float* const ub = &S.u[0][0][0][0];
    const int oi = (lx + 2) * FPZ + lz + 2;
    // halo point: x rows 0, 1, 18, 19 (threads 0..127), z columns 0, 1, 34, 35 (128..191)
    const bool halo = t < 192;
    int hrow = 0, hcol = 0;
    if (t < 128) {
        hrow = lx < 2 ? lx : FW + lx;
        hcol = lz + 2;
    } else if (halo) {
        hrow = ((t - 128) >> 2) + 2;
        hcol = (t & 3) < 2 ? (t & 3) : FZ + (t & 3);
    }
    const int hoff = max(0, min(nx - 1, x0 - 2 + hrow)) * sx + max(0, min(nz - 1, z0 - 2 + hcol));
    const int hi = hrow * FPZ + hcol;
    // closure windows (per-lane weights in increasing index; interior lanes put their 5-point
    // stencil at the end of the window)
    float wx[6], wz[6];
    int xb, zb;
    {
        const float wi[6] = {0.f, -D1C2, -D1C1, 0.f, D1C1, D1C2};
        const bool xlo = ix < nx - 1 - ix, zlo = iz < nz - 1 - iz;
        const int xr = xlo ? ix : max(0, nx - 1 - ix), zr = zlo ? iz : max(0, nz - 1 - iz);
        // (x rows of interior points start at row lx-1: row -1 for lx = 0 is not in the plane;
        // there the window starts at row 0 and the stencil at its start)
        const int sh = lx == 0 ? 1 : 0;
        xb = xr < 4 ? max(0, min(FPX - 6, xlo ? 2 - x0 : nx - 4 - x0)) : lx - 1 + sh;
        zb = zr < 4 ? (zlo ? 2 - z0 : nz - 4 - z0) : lz - 1;
#pragma unroll
        for (int k = 0; k < 6; k++) {
            wx[k] = xr >= 4 ? (sh ? (k < 5 ? wi[k + 1] : 0.f) : wi[k]) : (xlo ? c_d1w[xr][k] : -c_d1w[xr][5 - k]);
            wz[k] = zr >= 4 ? wi[k] : (zlo ? c_d1w[zr][k] : -c_d1w[zr][5 - k]);
        }
    }
    if (ZE) {
        // (values of weight zero may come from words never written)
        float* w = &S.pad[0];
        for (int k = t; k < (int)(sizeof(S) / sizeof(float)); k += FTHREADS) w[k] = 0.f;
        __syncthreads();
    }
    const float sn = uniform(fn.scale());
    const float ihx = uniform(1.0f / g.dx), ihy = uniform(1.0f / g.dy), ihz = uniform(1.0f / g.dz);
    const float fsx = uniform(sn * ihx), fsy = uniform(sn * ihy), fsz = uniform(sn * ihz);
    auto ld = [&](int f, int y, int off) {
        const unsigned i = (unsigned)((f % NC) * n3 + max(0, min(ny - 1, y)) * sy + off);
        return f < NC ? fn.code(i) : gld(lag, i);
    };
    float q[2 * NC][5], h[2 * NC];
#pragma unroll
    for (int f = 0; f < 2 * NC; f++) {
#pragma unroll
        for (int k = 0; k < 5; k++) q[f][k] = ld(f, ya - 2 + k, col);
        h[f] = halo ? ld(f, ya, hoff) : 0.f;
    }
    for (int o = ya; o < yb; o++) {
        float* const u = ub + (o & 1) * PL;
#pragma unroll
        for (int f = 0; f < 2 * NC; f++) {
            u[f * CP + oi] = q[f][2];
            if (halo) u[f * CP + hi] = h[f];
        }
        const unsigned p = (unsigned)(o * sy + col);
        const unsigned gi = (unsigned)((o * nx + ix) * nz + iz);
        if (outp) begin(p, gi);
        float qn[2 * NC];
#pragma unroll
        for (int f = 0; f < 2 * NC; f++) {
            qn[f] = ld(f, o + 3, col);
            if (halo) h[f] = ld(f, o + 1, hoff);
        }
        __syncthreads();
        if (outp) {
            float D[2 * NC][3];
#pragma unroll
            for (int f = 0; f < 2 * NC; f++) {
                const float* a = u + f * CP + oi;
                if (XE) {
                    const float* w = u + f * CP + xb * FPZ + lz + 2;
                    float v = wx[0] * w[0];
#pragma unroll
                    for (int k = 1; k < 6; k++) v += wx[k] * w[k * FPZ];
                    D[f][0] = v;
                } else {
                    D[f][0] = D1C1 * (a[FPZ] - a[-FPZ]) + D1C2 * (a[2 * FPZ] - a[-2 * FPZ]);
                }
                if (ZE) {
                    const float* w = u + f * CP + (lx + 2) * FPZ + zb;
                    float v = wz[0] * w[0];
#pragma unroll
                    for (int k = 1; k < 6; k++) v += wz[k] * w[k];
                    D[f][2] = v;
                } else {
                    D[f][2] = D1C1 * (a[1] - a[-1]) + D1C2 * (a[2] - a[-2]);
                }
                if (o >= 4 && o < ny - 4) {
                    D[f][1] = D1C1 * (q[f][3] - q[f][1]) + D1C2 * (q[f][4] - q[f][0]);
                } else {  // (a whole plane: a uniform branch)
                    const bool lo = o < 4;
                    const int r = lo ? o : ny - 1 - o;
                    float v = 0.f;
#pragma unroll 1
                    for (int k = 0; k < 6; k++) v += c_d1w[r][k] * ld(f, lo ? k : ny - 1 - k, col);
                    D[f][1] = lo ? v : -v;
                }
                D[f][0] *= f < NC ? fsx : ihx;
                D[f][1] *= f < NC ? fsy : ihy;
                D[f][2] *= f < NC ? fsz : ihz;
            }
            float F[3][NC], L[3][NC], fv[NC], lv[NC];
#pragma unroll
            for (int c = 0; c < NC; c++) {
                fv[c] = q[c][2] * sn;
                lv[c] = q[NC + c][2];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    F[k][c] = D[c][k];
                    L[k][c] = D[NC + c][k];
                }
            }
            end(gi, F, L, fv, lv);
        }
#pragma unroll
        for (int f = 0; f < 2 * NC; f++) {
#pragma unroll
            for (int k = 0; k < 4; k++) q[f][k] = q[f][k + 1];
            q[f][4] = qn[f];
        }
    }
}

// Acoustic event. Views of the slots itl-1, itl, itl+1 (a slot past the store has a null base
// and reads as zero); branch: 0 first sample, 1 middle, 2 last.
template <int FMT>
__global__ __launch_bounds__(FTHREADS) void acoustic_grad(SnapView<FMT> fm, SnapView<FMT> fn, SnapView<FMT> fp,
                                                          const float* __restrict__ adj, const float* __restrict__ K, Geom g,
                                                          ImagingTiles T, float sdt, int branch, double* __restrict__ gK,
                                                          double* __restrict__ gB) {
    __shared__ ImagingSmem<2> S;
    const float sm = uniform(fm.scale()), sp = uniform(fp.p ? fp.scale() : 0.f);
    const float w = uniform((branch == 0 ? 0.5f : 1.0f) * sdt);
    float k = 1.f, fmv = 0.f, fpv = 0.f;
    double ok = 0., ob = 0.;
    imaging_march<1, FMT>(
        S, fn, adj, g, T,
        [&](unsigned p, unsigned i) {
            k = gld(K, p);
            fmv = fm.code(p);
            fpv = fp.p ? fp.code(p) : 0.f;
            ok = gas(gK)[i];
            ob = gas(gB)[i];
        },
        [&](unsigned i, const float (&F)[3][1], const float (&L)[3][1], const float (&fv)[1], const float (&lv)[1]) {
            const float dot = L[0][0] * F[0][0] + L[1][0] * F[1][0] + L[2][0] * F[2][0];
            const float m = fmv * sm, n = fv[0], q = fpv * sp;
            const float d2t = branch == 1 ? q - 2.f * n + m : (branch == 0 ? q - n : -2.f * n + m);
            gas(gK)[i] = ok - (double)(1.0f / (sdt * k * k) * lv[0] * d2t);
            gas(gB)[i] = ob + (double)(w * dot);
        });
}

// Elastic / VTI event. `lag` is the adjoint field of the previous step (the reference uses
// the derivatives computed one step earlier); `adj` the current one (density term).
template <bool VTI, int FMT>
__global__ __launch_bounds__(FTHREADS) __attribute__((amdgpu_waves_per_eu(4)))
void elastic_grad(SnapView<FMT> fm, SnapView<FMT> fn, SnapView<FMT> fp, const float* __restrict__ adj,
                  const float* __restrict__ lag, EArgs A, ImagingTiles T, float sdt, int branch, double* __restrict__ gl,
                  double* __restrict__ gm, double* __restrict__ gr) {
    __shared__ ImagingSmem<6> S;
    const Geom g = A.g;
    const float sm = uniform(fm.scale()), sp = uniform(fp.p ? fp.scale() : 0.f);
    const float w = uniform((branch == 0 ? 0.5f : 1.0f) * sdt), isdt = uniform(1.0f / sdt);
    float av[3] = {0.f, 0.f, 0.f}, fmv[3] = {0.f, 0.f, 0.f}, fpv[3] = {0.f, 0.f, 0.f};
    float U = 1.f, C = 1.f, E = 0.f, C13 = 1.f, C66 = 1.f;
    double ol = 0., om = 0., orr = 0.;
    imaging_march<3, FMT>(
        S, fn, lag, g, T,
        [&](unsigned p, unsigned i) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const unsigned q = c * g.n + p;
                av[c] = gld(adj, q);
                fmv[c] = fm.code(q);
                fpv[c] = fp.p ? fp.code(q) : 0.f;
            }
            if (VTI) {
                C = gld(A.lam, p); U = gld(A.mu, p); E = gld(A.eps, p); C13 = gld(A.c13, p); C66 = gld(A.c66, p);
            }
            ol = gas(gl)[i];
            om = gas(gm)[i];
            orr = gas(gr)[i];
        },
        [&](unsigned i, const float (&F)[3][3], const float (&Aj)[3][3], const float (&fv)[3], const float (&)[3]) {
            // forward-field terms named as in the reference: temp[0..8]
            const float t0 = F[0][0], t1 = F[1][1], t2 = F[2][2], t3 = F[0][2], t4 = F[2][0], t5 = F[0][1], t6 = F[1][0],
                        t7 = F[1][2], t8 = F[2][1];
            float gL, gM;
            if (!VTI) {
                gL = w * (Aj[0][0] + Aj[1][1] + Aj[2][2]) * (t0 + t1 + t2);
                gM = w * ((Aj[2][0] + Aj[0][2]) * (t3 + t4) + (Aj[1][0] + Aj[0][1]) * (t5 + t6) +
                          (Aj[2][1] + Aj[1][2]) * (t7 + t8) + 2.f * Aj[0][0] * t0 + 2.f * Aj[1][1] * t1 +
                          2.f * Aj[2][2] * t2);
            } else {
                const float del = ((C13 + U) * (C13 + U) - (C + U) * (C + U)) / (2.f * (C + U) * (C + 2.f * U));
                const float gam = (C66 - U) / (2.f * U);
                const float v1 = sqrtf(2.f * (C + 2.f * U) * (C + U) * del + (C + U) * (C + U));
                const float v2 = ((1.f + 2.f * del) * C + (1.f + 3.f * del) * U) / v1;
                const float v3 = ((1.f + 3.f * del) * C + (1.f + 4.f * del) * U) / v1 - 1.f;
                const float v4 = (Aj[0][0] + Aj[1][1]) * t2 + Aj[2][2] * (t0 + t1);
                gL = w * ((1.f + 2.f * E) * (Aj[0][0] + Aj[1][1]) * (t0 + t1) + Aj[2][2] * t2 + v2 * v4);
                gM = w * (2.f * (1.f + 2.f * E) * (Aj[0][0] * t0 + Aj[1][1] * t1) + 2.f * Aj[2][2] * t2 +
                          4.f * (E - gam) * (Aj[0][0] * t1 + Aj[0][0] * t0) + (Aj[1][2] + Aj[2][1]) * (t7 + t8) +
                          (Aj[0][2] + Aj[2][0]) * (t3 + t4) + (1.f + 2.f * gam) * (Aj[0][1] + Aj[1][0]) * (t5 + t6) + v3 * v4);
            }
            float rt = 0.f;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float m = fmv[c] * sm, n = fv[c], q = fpv[c] * sp;
                rt += av[c] * (branch == 1 ? q - 2.f * n + m : (branch == 0 ? q - n : -n + m));
            }
            gas(gl)[i] = ol + (double)gL;
            gas(gm)[i] = om + (double)gM;
            gas(gr)[i] = orr + (double)(isdt * rt);
        });
}

}  // namespace fwi3d
