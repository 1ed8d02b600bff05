// One-launch acoustic time step (gfx950): every point of nl_we_op_a::propagate
// (src/cpp/we_op.cpp:1662-1791), closure rows, SATs, absorbing scaling and taper included,
// with the receivers of the step and its source injection.
//
// Workgroups of 32 z x 16 x points (512 threads) march along y over a chunk of planes: u and
// 1/rho of the column in register queues along y, of the plane in two LDS planes with 2-cell
// halos (one barrier per plane). Near a face the operator along its normal, D2 closure row and
// SAT, is 8 time-invariant coefficients per point on the 8 values from the face (acoustic_tables,
// formed once per propagation): along x and z from the LDS plane (tiles are laid so that a
// face's rows and their stencils lie in one tile), along y from memory, a whole plane at a time.
// With the rows' and SATs' own arithmetic instead (its divisions and scattered constants, one
// branch per row and face) a plane took 4.4 us, with the coefficients 1.2 us.
//
// Small grids are bound by the latency of a plane (load, barrier, update) times the planes of
// a chunk, so the chunk is as short as fills the chip; large ones by HBM (20 B per cell).
// Per step with its injection (HIP events around graph replays): (ny, nx, nz) = (40, 52, 47) 6.7 us,
// 100^3 16.6, 128^3 20, (203, 187, 211) 53.5 (3.0 TB/s of the 20 B; 79 VGPRs, three workgroups per
// CU; the issue slots are about half used), against 13, 21.6, 29 and 65 us with interior tiles, a
// point-wise shell and an injection launch.
//
// Injection. A word of mask and one of rank per 32 points mark the points that sources touch
// (0.25 B per cell); a marked point adds its contributions, which the previous step's launch
// formed (V: one value per contribution, two steps' worth), in the order of the lists. As a
// launch of its own the injection took 4 to 6 us of each step, however few the sources.
#pragma once
#include "fused.hpp"

namespace fwi3d {

// Boundary data. Coefficients of 6 rows from each face, 2 float4 an entry, counted from the face:
//   zc[((face ny + y) nx + x) 6 + row], xc[((face ny + y) 6 + row) nz + z],
//   yc[((face 6 + row) nx + x) nz + z]; of d2/h^2 plus the SATs of that face.
// Face points, {sum over the point's absorbing faces of impedance / (h H0 dt), 1 / scaling}:
//   zf[(face ny + y) nx + x], xf[(face ny + y) nz + z], yf[(face nx + x) nz + z].
struct AcuTabs {
    const float4 *zc, *xc, *yc;
    const float2 *zf, *xf, *yf;
};
inline size_t acoustic_tables_bytes(const Geom& g) {
    return ((size_t)g.ny * g.nx + (size_t)g.ny * g.nz + (size_t)g.nx * g.nz) * (24 * sizeof(float4) + 2 * sizeof(float2));
}
inline AcuTabs acoustic_tabs(float4* base, const Geom& g) {
    const size_t a = (size_t)g.ny * g.nx, b = (size_t)g.ny * g.nz, c = (size_t)g.nx * g.nz;
    AcuTabs t;
    t.zc = base;
    t.xc = t.zc + 24 * a;
    t.yc = t.xc + 24 * b;
    t.zf = (const float2*)(t.yc + 24 * c);
    t.xf = t.zf + 2 * a;
    t.yf = t.xf + 2 * b;
    return t;
}
// One thread per (face, point of the face): its 6 rows and its face point.
__global__ __launch_bounds__(256) void acoustic_tables(AcuArgs A, AcuTabs T) {
    const Geom g = A.g;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    long long q = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long a = 2LL * ny * nx, b = 2LL * ny * nz, c = 2LL * nx * nz;
    if (q >= a + b + c) return;
    int ax, hi, ix = 0, iy = 0, iz = 0;  // ax 0: z, 1: x, 2: y
    float4* row;
    float2* face;
    int rstride;  // entries between rows
    if (q < a) {
        ax = 0;
        ix = (int)(q % nx); iy = (int)(q / nx % ny); hi = (int)(q / nx / ny);
        row = (float4*)T.zc + q * 12;
        rstride = 1;
        face = (float2*)T.zf + q;
    } else if ((q -= a) < b) {
        ax = 1;
        iz = (int)(q % nz); iy = (int)(q / nz % ny); hi = (int)(q / nz / ny);
        row = (float4*)T.xc + ((q / nz) * 6 * nz + iz) * 2;
        rstride = nz;
        face = (float2*)T.xf + q;
    } else {
        q -= b;
        ax = 2;
        iz = (int)(q % nz); ix = (int)(q / nz % nx); hi = (int)(q / nz / nx);
        row = (float4*)T.yc + ((long long)hi * 6 * nx * nz + (q - (long long)hi * nx * nz)) * 2;
        rstride = nx * nz;
        face = (float2*)T.yf + q;
    }
    const int len = ax == 0 ? nz : (ax == 1 ? nx : ny), st = ax == 0 ? 1 : (ax == 1 ? g.sx : g.sy);
    const float h = ax == 0 ? g.dz : (ax == 1 ? g.dx : g.dy), ih2 = 1.0f / (h * h);
    const int e = hi ? len - 1 : 0;
    if (ax == 0) iz = e;
    else if (ax == 1) ix = e;
    else iy = e;
    const int p = g.at(ix, iy, iz), bc = A.bc[2 * ax + hi];
    float bb[8], w[8];
#pragma unroll
    for (int k = 0; k < 8; k++) bb[k] = gld(A.b, p + (hi ? -k : k) * st);
#pragma unroll 1
    for (int r = 0; r < 6; r++) {
        d2_coefs(r, bb, w);
#pragma unroll
        for (int k = 0; k < 8; k++) w[k] *= ih2;
        if (bc == 1 && r < 4) {
            w[0] += ih2 / c_hnorm[r] * c_sat_s[r] * bb[0];
            if (r == 0) w[0] -= bb[0] * ih2 / (A.alpha * SAT_H0);
        } else if (bc != 0 && r == 0) {
#pragma unroll
            for (int k = 0; k < 4; k++) w[k] -= ih2 / SAT_H0 * bb[0] * c_sat_s[k];
        }
        row[2LL * r * rstride] = make_float4(w[0], w[1], w[2], w[3]);
        row[2LL * r * rstride + 1] = make_float4(w[4], w[5], w[6], w[7]);
    }
    const float Kp = A.K[p], imp = 0.5f / sqrtf(Kp / bb[0]) / A.dt;
    float s = 0.f;
    if ((iz == 0 && A.bc[0] == 2)) s += imp / (SAT_H0 * g.dz);
    if ((iz == nz - 1 && A.bc[1] == 2)) s += imp / (SAT_H0 * g.dz);
    if ((ix == 0 && A.bc[2] == 2)) s += imp / (SAT_H0 * g.dx);
    if ((ix == nx - 1 && A.bc[3] == 2)) s += imp / (SAT_H0 * g.dx);
    if ((iy == 0 && A.bc[4] == 2)) s += imp / (SAT_H0 * g.dy);
    if ((iy == ny - 1 && A.bc[5] == 2)) s += imp / (SAT_H0 * g.dy);
    *face = make_float2(s, 1.f / acu_scale(g, A.bc, Kp, bb[0], ix, iy, iz, A.dt));
}

struct AcuTiles { int ntz, ntx, nyc, chunk; AcuTabs tab; };
// Planes per workgroup: as few as keep the workgroups within one round of the chip (three on each
// of 256 CUs), at most 6 (on large grids, where several rounds run anyway, 5 to 10 measured alike and
// 3 and 16 slower). chunk > 0: by hand (any count: past ny it is the whole axis).
inline AcuTiles acoustic_tiles(const Geom& g, int chunk) {
    AcuTiles T{};
    T.ntz = fused_tile_count(g.nz, FZ);
    T.ntx = fused_tile_count(g.nx, FW);
    const int fit = std::max(1, 768 / (T.ntz * T.ntx));
    T.chunk = std::min(g.ny, chunk > 0 ? chunk : std::min(6, (g.ny + fit - 1) / fit));
    T.nyc = (g.ny + T.chunk - 1) / T.chunk;
    return T;
}
// Tile that outputs point i of an axis (fused_tile).
__device__ __forceinline__ int fused_tile_of(int n, int w, int nt, int i) {
    return i >= (nt == 1 ? 0 : (n < w + 8 ? 8 : n - w)) ? nt - 1 : i / w;
}

struct AcuSmem {
    float u[2][FPX][FPZ], b[2][FPX][FPZ];  // plane mod 2, x row (from x0-2), z column (from z0-2)
};

// Source points in the step kernels: flag[(y ntx + tx) ntz + tz], the tile outputs injected
// points of plane y; mask[p / 32] = {bit p % 32 set: injected, slot of the word's first marked
// point}; perm: slot -> target; V: the values of step k at (k & 1) * nv.
struct InjMap {
    const int* flag;
    const uint2* mask;
    const int* perm;
    float* V;
    int nv;
};

// Sum of the injection at point p onto val, in the order of the list; scale: the last taper factor,
// which the values lack. Four loads are in flight: with one at a time a plane of 4 receivers per
// point (100^3, adjoint) took 76 us per step, now 39; a launch of its own takes 57.
__device__ __forceinline__ float inject_at(const InjMap& M, const InjTab& I, unsigned p, int k, float scale, float val) {
    const unsigned bit = p & 31u;
    const GAS unsigned* word = gas((const unsigned*)M.mask) + 2 * (p >> 5);
    const uint2 w = make_uint2(word[0], word[1]);
    if (!((w.x >> bit) & 1u)) return val;
    const int j = gas(M.perm)[w.y + __popc(w.x & ((1u << bit) - 1u))];
    const int e1 = gas(I.tbeg)[j + 1];
    const float* V = M.V + (size_t)(k & 1) * M.nv;
    int e = gas(I.tbeg)[j];
    for (; e + 4 <= e1; e += 4) {
        const float v0 = gas(V)[e], v1 = gas(V)[e + 1], v2 = gas(V)[e + 2], v3 = gas(V)[e + 3];
        val = __builtin_fmaf(v3, scale, __builtin_fmaf(v2, scale, __builtin_fmaf(v1, scale, __builtin_fmaf(v0, scale, val))));
    }
    for (; e < e1; e++) val = __builtin_fmaf(gas(V)[e], scale, val);
    return val;
}

// Contribution e of step k's injection, without the taper's last factor (along y).
__device__ __forceinline__ void acoustic_inj_value(const AcuArgs& A, const InjTab& I, const InjMap& M,
                                                   const float* __restrict__ src, int nt, int k, int e) {
    if (e >= M.nv) return;
    int r, a, bb, c, de, ix, iy, iz;
    inj_decode(I, I.tlst[e], r, a, bb, c, de);
    inj_point(I, r, a, bb, c, de, ix, iy, iz);
    const int p = A.g.at(ix, iy, iz);
    const float v = inj_value(I, src, nt, k, 0, r, a, bb, c, de);
    float add = A.dt * A.dt * v * A.K[p];
    add = add / acu_scale(A.g, A.bc, A.K[p], A.b[p], ix, iy, iz, A.dt);
    M.V[(size_t)(k & 1) * M.nv + e] = (add * gld(A.tz2, iz)) * gld(A.tx2, ix);
}

// EDGE: the tile may hold x / z closure rows and face points.
template <bool EDGE>
__device__ __forceinline__ void acoustic_fused_tile(const AcuArgs& A, const AcuTiles& T, const InjTab& I, const InjMap& M,
                                                    int k, int l, AcuSmem& S) {
    const Geom& g = A.g;
    const int nx = g.nx, ny = g.ny, nz = g.nz, sx = g.sx, sy = g.sy;
    const float idx2 = 1.0f / (g.dx * g.dx), idy2 = 1.0f / (g.dy * g.dy), idz2 = 1.0f / (g.dz * g.dz);
    const int tz = l % T.ntz, tx = (l / T.ntz) % T.ntx, ch = l / (T.ntz * T.ntx);
    const int ya = ch * T.chunk, yb = min(ny, ya + T.chunk);
    int z0, zo0, zo1, x0, xo0, xo1;
    fused_tile(nz, FZ, tz, T.ntz, z0, zo0, zo1);
    fused_tile(nx, FW, tx, T.ntx, x0, xo0, xo1);
    const int t = threadIdx.x;
    const int lz = t & (FZ - 1), lx = t >> 5;
    const int ix = x0 + lx, iz = z0 + lz;
    const int cx = min(ix, nx - 1), cz = min(iz, nz - 1);
    const int col = cx * sx + cz;
    const bool outp = ix >= xo0 && ix < xo1 && iz >= zo0 && iz < zo1;
    const int oi = (lx + 2) * FPZ + lz + 2;
    // distance from the nearer face, and from it inwards: first LDS word and step
    const bool xlo = ix < nx - 1 - ix, zlo = iz < nz - 1 - iz;
    const int xr = !EDGE ? 8 : (xlo ? ix : max(0, nx - 1 - ix)), zr = !EDGE ? 8 : (zlo ? iz : max(0, nz - 1 - iz));
    const int xs = xlo ? FPZ : -FPZ, zs = zlo ? 1 : -1;
    const int xb = oi - xr * xs, zb = oi - zr * zs;
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
    auto ld = [&](const float* __restrict__ f, int y, int off) { return gld(f, (unsigned)(max(0, min(ny - 1, y)) * sy + off)); };
    float u[6], b[5], hu = 0.f, hb = 0.f;  // u at o-2..o+3, 1/rho at o-1..o+3
    float p1, p2[2];                       // D2 pairs along y: p1 from o-1, p2 from o-2 and o-1
#pragma unroll
    for (int q = 0; q < 5; q++) u[q] = ld(A.curr, ya - 2 + q, col);
#pragma unroll
    for (int q = 0; q < 4; q++) b[q] = ld(A.b, ya - 1 + q, col);
    {
        const float bm2 = ld(A.b, ya - 2, col);
        p1 = d2_pair1(bm2, b[0], b[1], b[2]);
        p2[0] = d2_pair2(bm2, b[0], b[1]);
        p2[1] = d2_pair2(b[0], b[1], b[2]);
    }
    if (halo) {
        hu = ld(A.curr, ya, hoff);
        hb = ld(A.b, ya, hoff);
    }
    const float tzx = gld(A.tz2, cz) * gld(A.tx2, cx);
    // the 8 products of a row near a face: words from f in steps of st
    auto row8 = [](float4 a, float4 b, const auto& f) {
        return a.x * f(0) + a.y * f(1) + a.z * f(2) + a.w * f(3) + b.x * f(4) + b.y * f(5) + b.z * f(6) + b.w * f(7);
    };
    unsigned long long flags = 0;
    for (int o = ya; o < yb; o++) {
        float *const su = &S.u[o & 1][0][0], *const sb = &S.b[o & 1][0][0];
        su[oi] = u[2];
        sb[oi] = b[1];
        if (halo) {
            su[hi] = hu;
            sb[hi] = hb;
        }
        const unsigned p = (unsigned)(o * sy + col);
        u[5] = ld(A.curr, o + 3, col);
        b[4] = ld(A.b, o + 3, col);
        float pv = gld(A.prev, p);
        const float Kp = gld(A.K, p);
        // (flags of the next 64 planes, one per lane: a scalar load per plane would make the
        // LDS waits wait for it)
        if (M.flag && ((o - ya) & 63) == 0) {
            const int y = o + (t & 63);
            flags = __ballot(y < yb && gas(M.flag)[(y * T.ntx + tx) * T.ntz + tz] != 0);
        }
        const bool inj = (flags >> ((o - ya) & 63)) & 1;
        if (halo) {
            hu = ld(A.curr, o + 1, hoff);
            hb = ld(A.b, o + 1, hoff);
        }
        const float tfy = gld(A.ty2, o);
        // (uniform: a plane near a y face, its distance from it)
        const bool ylo = o < ny - 1 - o;
        const int yr = ylo ? o : ny - 1 - o;
        float4 tz0{}, tz1{}, tx0{}, tx1{};
        float ydot = 0.f;
        float2 fe = make_float2(0.f, 1.f);
        if (EDGE && zr < 6) {
            const unsigned e = ((((zlo ? 0 : ny) + o) * nx + cx) * 6 + zr) * 32u;
            tz0 = gld4(T.tab.zc, e);
            tz1 = gld4(T.tab.zc, e + 16);
        }
        if (EDGE && xr < 6) {
            const unsigned e = ((((xlo ? 0 : ny) + o) * 6 + xr) * nz + cz) * 32u;
            tx0 = gld4(T.tab.xc, e);
            tx1 = gld4(T.tab.xc, e + 16);
        }
        if (yr < 6) {
            const unsigned e = ((((ylo ? 0 : 6) + yr) * nx + cx) * nz + cz) * 32u;
            const int py = (ylo ? 0 : ny - 1) * sy + col, ys = ylo ? sy : -sy;
            ydot = row8(gld4(T.tab.yc, e), gld4(T.tab.yc, e + 16), [&](int j) { return gld(A.curr, py + j * ys); });
        }
        if (min(min(xr, zr), yr) == 0) {
            const float2* f = zr == 0 ? T.tab.zf + (((zlo ? 0 : ny) + o) * nx + cx)
                                      : (xr == 0 ? T.tab.xf + (((xlo ? 0 : ny) + o) * nz + cz)
                                                 : T.tab.yf + (((ylo ? 0 : nx) + cx) * nz + cz));
            fe.x = gas((const float*)f)[0];
            fe.y = gas((const float*)f)[1];
        }
        const float q1 = d2_pair1(b[0], b[1], b[2], b[3]), q2 = d2_pair2(b[1], b[2], b[3]);
        __syncthreads();
        if (outp) {
            float dx, dz, lap;
            if (!EDGE || xr >= 6)
                dx = idx2 * D2W(sb[oi - 2 * FPZ], sb[oi - FPZ], b[1], sb[oi + FPZ], sb[oi + 2 * FPZ])(
                                su[oi - 2 * FPZ], su[oi - FPZ], u[2], su[oi + FPZ], su[oi + 2 * FPZ]);
            else
                dx = row8(tx0, tx1, [&](int j) { return su[xb + j * xs]; });
            if (!EDGE || zr >= 6)
                dz = idz2 * D2W(sb[oi - 2], sb[oi - 1], b[1], sb[oi + 1], sb[oi + 2])(su[oi - 2], su[oi - 1], u[2], su[oi + 1],
                                                                                     su[oi + 2]);
            else
                dz = row8(tz0, tz1, [&](int j) { return su[zb + j * zs]; });
            lap = yr >= 6 ? idy2 * D2W(p2[0], p1, q1, q2)(u[0], u[1], u[2], u[3], u[4]) : ydot;
            lap += dx + dz;
            const float tf = tzx * tfy;
            if (A.prev_tapered) pv *= tf;
            float nv = A.dt2 * Kp * (lap + fe.x * pv) + (2.f * u[2] - pv);
            nv *= fe.y * tf;
            if (inj) nv = inject_at(M, I, p, k, tfy, nv);
            gst(A.next, p, nv);
        }
        p2[0] = p2[1];
        p2[1] = q2;
        p1 = q1;
#pragma unroll
        for (int q = 0; q < 5; q++) u[q] = u[q + 1];
#pragma unroll
        for (int q = 0; q < 4; q++) b[q] = b[q + 1];
    }
}

// ---- the source map of a shot: mark the targets' points, number the marked points of each
// word, list the targets by number (three launches over n / 32 words or the targets)
__device__ __forceinline__ unsigned inj_target_point(const Geom& g, const InjTab& I, int j) {
    int r, a, bb, c, de, ix, iy, iz;
    inj_decode(I, I.tlst[I.tbeg[j]], r, a, bb, c, de);
    inj_point(I, r, a, bb, c, de, ix, iy, iz);
    return (unsigned)g.at(ix, iy, iz);
}
__global__ __launch_bounds__(256) void inj_map_clear(uint2* mask, int nw, int* flag, int nf, int* count) {
    const int w = blockIdx.x * 256 + threadIdx.x;
    if (w < nw) mask[w] = make_uint2(0u, 0u);
    if (w < nf) flag[w] = 0;
    if (w == 0) *count = 0;
}
__global__ __launch_bounds__(256) void inj_map_mark(uint2* mask, int* flag, int ntz, int ntx, InjTab I, Geom g) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= I.ntgt) return;
    const unsigned p = inj_target_point(g, I, j), q = p % (unsigned)g.sy;
    const int iy = (int)(p / (unsigned)g.sy), ix = (int)(q / (unsigned)g.sx), iz = (int)(q % (unsigned)g.sx);
    atomicOr(&mask[p >> 5].x, 1u << (p & 31u));
    flag[(iy * ntx + fused_tile_of(g.nx, FW, ntx, ix)) * ntz + fused_tile_of(g.nz, FZ, ntz, iz)] = 1;
}
__global__ __launch_bounds__(256) void inj_map_number(uint2* mask, int nw, int* count) {
    const int w = blockIdx.x * 256 + threadIdx.x;
    if (w < nw && mask[w].x) mask[w].y = (unsigned)atomicAdd(count, __popc(mask[w].x));
}
__global__ __launch_bounds__(256) void inj_map_list(const uint2* mask, InjTab I, Geom g, int* perm) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= I.ntgt) return;
    const unsigned p = inj_target_point(g, I, j);
    const uint2 w = mask[p >> 5];
    perm[w.y + __popc(w.x & ((1u << (p & 31u)) - 1u))] = j;
}

}  // namespace fwi3d
