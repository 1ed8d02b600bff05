// Fused elastic / VTI time step (gfx950): one launch computes one time step of
// nl_we_op_e::propagate (src/cpp/we_op.cpp:646-836) / nl_we_op_vti::propagate
// (we_op.cpp:1290-1497) at every point, including the closure rows, the traction SATs and
// the absorbing scaling of the six faces, with the normal stresses and shear fluxes formed
// on chip: no flux buffer travels through HBM.
//
// Tile: 32 z points (one 128-byte line per row) x 16 x rows, 512 threads (a wave holds two x
// rows). A workgroup of the planes [6, ny-6) marches along y over a chunk of planes
// (FusedTile::march): a ring of six LDS planes holds u (2-cell halos) at o-2..o+3, so that
// every derivative of u, along y too and at the halo points, reads LDS; the fluxes that are
// differentiated along x and z at plane o go to LDS planes, those differentiated along y
// (T_y, F_yx, F_yz) are formed at plane o+2 into register queues. Halo fluxes are formed by
// the first 192 threads (128 points of four x-halo rows, 64 of four z-halo columns); their D1
// reaches two cells further (e0, e1). A workgroup of a y face (FusedTile::yface) holds planes
// 0..5 from the face in the ring.
//
// Occupancy: u in LDS instead of register queues leaves 104 VGPRs (VTI 125) for the middle
// tiles, so two workgroups share a CU (70 / 75 KB of LDS each) and hide each other's two
// barriers per plane. With the y neighbours in register queues and four ring planes (one
// barrier per plane) VTI took 158 VGPRs, one workgroup per CU: 102 against 72 us for the
// middle tiles of (nz, nx, ny) = (200, 160, 160).
//
// Closure rows read time-invariant coefficients (closures.hpp), so that all rows run one
// code: along x whole waves (two x rows each), along z the lanes of a wave with a window of 6
// or 8 points and per-lane weights. With a row switch over register copies of the operands
// the edge tiles took 185 VGPRs and one workgroup per CU: 144 us of the elastic step at
// 200^3, now 94 us as a launch of its own.
//
// All tiles are one launch. Steps with their injection launch of 5 to 6 us (MI355X, HIP events,
// the chunks of fused_plan): elastic 200^3 196 us (191 the step's launch alone, by a kernel trace;
// 187 with the autotuner's chunks), against 253 us, without injection, where the y faces are left to
// a flux pass and slab kernels (82 us alone) and the edge tiles are a launch on a second stream; 256^3
// 312 against 437 us; (ny, nx, nz) = (61, 75, 68) 37 against 90 us; VTI (160, 160, 200) 190 against
// 282 us, (150, 144, 71) 92 (81 with the autotuner's chunks) against 141 us. What bounds it: HBM traffic
// and vector issue together (middle tiles alone: 5.1 TB/s of measured traffic, the rate of a
// plain copy, and 55 % of the issue slots).
//
// Tiling of an axis of n points into tiles of w (fused_tile): tiles at multiples of w
// whose outputs stop at n - w, then a last tile at n - w with the rest, so that the
// closure rows of each face and the points their stencils read lie inside one tile
// (tile 0 outputs at least [0, 8), the last tile [n-8, n)).
#pragma once
#include "closures.hpp"
#include "elastic.hpp"

namespace fwi3d {

constexpr int FZ = 32;                 // z points per tile
constexpr int FW = 16;                 // x rows per tile
constexpr int FPZ = FZ + 4, FPX = FW + 4;
constexpr int FTHREADS = FZ * FW;      // 512
constexpr int FRING = 6;               // planes o-2..o+3 of u in LDS

// D1 closure rows by LDS / row index: weights of the 6 points nearest a low face.
static __constant__ float c_d1w[4][6] = {
    {(float)kD1Closure[0][0], (float)kD1Closure[0][1], (float)kD1Closure[0][2], (float)kD1Closure[0][3], 0.f, 0.f},
    {(float)kD1Closure[1][0], 0.f, (float)kD1Closure[1][2], 0.f, 0.f, 0.f},
    {(float)kD1Closure[2][0], (float)kD1Closure[2][1], 0.f, (float)kD1Closure[2][3], (float)kD1Closure[2][4], 0.f},
    {(float)kD1Closure[3][0], 0.f, (float)kD1Closure[3][2], 0.f, (float)kD1Closure[3][4], (float)kD1Closure[3][5]},
};

// Rows of D1 over the 8 planes from a y face: 0-3 the closure, 4 and 5 interior stencils.
struct Y1W { float w[6][8]; __host__ __device__ constexpr const float* operator[](int r) const { return w[r]; } };
constexpr Y1W make_y1w() {
    Y1W t{};
    for (int r = 0; r < 6; r++)
        for (int j = 0; j < 8; j++) {
            const int m = j - r;
            t.w[r][j] = r < 4 ? (j < 6 ? (float)kD1Closure[r][j] : 0.f)
                              : (m == 1 ? (float)kD1Int[0] : (m == -1 ? -(float)kD1Int[0] : (m == 2 ? (float)kD1Int[1] : (m == -2 ? -(float)kD1Int[1] : 0.f))));
        }
    return t;
}
static __constant__ Y1W c_y1w = make_y1w();

// Workgroups of the step, by class: corner tiles (first or last tile along both x and z),
// side tiles (the other tiles at an x or z face), the tiles of the 6 planes at each y face,
// middle tiles. A march class has n[c] = tiles x y chunks of chunk[c] planes.
enum { FC_CORNER = 0, FC_SIDE = 1, FC_YFACE = 2, FC_MID = 3, FC_N = 4 };
struct FusedTiles {
    int ntz, ntx;
    int ya, yb;          // planes of the march classes: [6, ny-6)
    int n[FC_N], chunk[FC_N];
    ClosureTabs tab;     // boundary data
    const float* rdt;    // dt^2 / rho
};

__host__ __device__ inline int fused_tile_count(int n, int w) {
    if (n <= w) return 1;
    if (n < w + 8) return 2;
    return (n - w + w - 1) / w + 1;
}
// Origin and output range [o0, o1) of tile t of nt.
__host__ __device__ inline void fused_tile(int n, int w, int t, int nt, int& org, int& o0, int& o1) {
    if (n <= w) {
        org = 0; o0 = 0; o1 = n;
        return;
    }
    if (t == nt - 1) {
        org = n - w; o0 = n < w + 8 ? 8 : n - w; o1 = n;
        return;
    }
    org = w * t; o0 = w * t;
    o1 = n < w + 8 ? 8 : (w * t + w < n - w ? w * t + w : n - w);
}

template <bool VTI>
struct FusedSmem {
    static constexpr int NB = VTI ? 3 : 1;
    float pad[8];              // (a z window of an edge tile may start one point before u)
    float u[FRING][3][FPX][FPZ];  // ring slot (plane mod 6), component, x row (from x0-2), z column (from z0-2)
    // plane o:
    float b[NB][FPX][FPZ];     // D2 coefficient fields: mu [, c66, c11b]
    float tx[FPX][FZ];         // T (elastic) / T_x (VTI), own and x-halo rows
    float tz[FW][FPZ];         // T / T_z, own and z-halo columns
    float fxy[FPX][FZ], fxz[FPX][FZ];
    float fzx[FW][FPZ], fzy[FW][FPZ];
    float wd1[8][6];           // D1 closure rows along x: 0-3 at a low face, 4-7 at a high face, increasing x
};

// D1 at an interior point, the spacing folded into the two weights.
struct D1W {
    float k1, k2;
    __device__ __forceinline__ D1W(float ih) : k1(uniform(D1C1 * ih)), k2(uniform(D1C2 * ih)) {}
    __device__ __forceinline__ float operator()(float m2, float m1, float p1, float p2) const {
        return k1 * (p1 - m1) + k2 * (p2 - m2);
    }
    __device__ __forceinline__ float add(float a, float m2, float m1, float p1, float p2) const {
        return k2 * (p2 - m2) + (k1 * (p1 - m1) + a);
    }
};
// Interior D2(b) (times h^2): the operator couples point i to i+1 by p1(b) and to i+2 by
// p2(b), symmetrically, and its row sums vanish (spatial_operators.hpp:37), so the weights
// of a point are p1 and p2 of the four pairs it belongs to, and minus their sum.
__device__ __forceinline__ float d2_pair1(float bm1, float b0, float bp1, float bp2) {
    return D2C5 * (b0 + bp1) + D2C6 * (bm1 + bp2);
}
__device__ __forceinline__ float d2_pair2(float b0, float bp1, float bp2) { return D2C8 * bp1 + D2C7 * (b0 + bp2); }
struct D2W {
    float m2, m1, p1, p2, c0;
    __device__ __forceinline__ D2W(float m2_, float m1_, float p1_, float p2_)
        : m2(m2_), m1(m1_), p1(p1_), p2(p2_), c0(-((m1_ + p1_) + (m2_ + p2_))) {}
    __device__ __forceinline__ D2W(float bm2, float bm1, float b0, float bp1, float bp2)
        : D2W(d2_pair2(bm2, bm1, b0), d2_pair1(bm2, bm1, b0, bp1), d2_pair1(bm1, b0, bp1, bp2), d2_pair2(b0, bp1, bp2)) {}
    __device__ __forceinline__ float operator()(float um2, float um1, float u0, float up1, float up2) const {
        return c0 * u0 + m1 * um1 + p1 * up1 + m2 * um2 + p2 * up2;
    }
};

// Tile classes: the tiles away from the x and z faces (the middle tiles of both axes,
// whose outputs, and the fluxes and stencils they read, are at least 14 points inside
// those faces) run a body without closure rows and face terms, the side tiles one with
// those of their axis, the corner tiles one with both. Side tiles: those of the first and
// last x columns of tiles, then those of the first and last z tiles.
__host__ __device__ inline int fused_middle_tiles(int ntz, int ntx) {
    return (ntz < 3 || ntx < 3) ? 0 : (ntz - 2) * (ntx - 2);
}
__host__ __device__ inline int fused_corner_tiles(int ntz, int ntx) {
    return (ntz == 1 ? 1 : 2) * (ntx == 1 ? 1 : 2);
}
__host__ __device__ inline int fused_side_tiles(int ntz, int ntx) {
    return (ntx == 1 ? 1 : 2) * (ntz > 2 ? ntz - 2 : 0) + (ntz == 1 ? 1 : 2) * (ntx > 2 ? ntx - 2 : 0);
}
// Corner tile c: (tz, tx) packed as tz | tx << 16.
__device__ __forceinline__ int fused_corner_tile(int c, int ntz, int ntx) {
    const int nzc = ntz == 1 ? 1 : 2;
    return ((c % nzc) == 0 ? 0 : ntz - 1) | (((c / nzc) == 0 ? 0 : ntx - 1) << 16);
}
// Side tile e: the x-edge columns' tiles between the corners, then the z-edge rows'.
__device__ __forceinline__ int fused_side_tile(int e, int ntz, int ntx) {
    const int mz = ntz > 2 ? ntz - 2 : 0, nxs = (ntx == 1 ? 1 : 2) * mz;
    const int mz1 = mz > 0 ? mz : 1, mx = ntx > 2 ? ntx - 2 : 1, f = e - nxs;
    const int tz = e < nxs ? 1 + e % mz1 : (f / mx == 0 ? 0 : ntz - 1);
    const int tx = e < nxs ? (e / mz1 == 0 ? 0 : ntx - 1) : 1 + f % mx;
    return tz | (tx << 16);
}

// Workgroup l of a shot's step -> class and item. Workgroups l = x (mod 8) run on one XCD:
// it takes the x-th eighth of every class, so that the tiles of an XCD are neighbours (their
// halos meet in its L2) and every XCD has the same mix of classes.
__host__ __device__ inline int fused_workgroups(const FusedTiles& F) {
    int most = 0;
    for (int x = 0; x < 8; x++) {
        int k = 0;
        for (int c = 0; c < FC_N; c++) k += (((x + 1) * F.n[c]) >> 3) - ((x * F.n[c]) >> 3);
        most = k > most ? k : most;
    }
    return 8 * most;
}
__device__ __forceinline__ bool fused_item(const FusedTiles& F, int l, int& cls, int& item) {
    const int x = l & 7;
    int k = l >> 3;
#pragma unroll
    for (int c = 0; c < FC_N; c++) {
        const int b = (x * F.n[c]) >> 3, e = ((x + 1) * F.n[c]) >> 3;
        if (k < e - b) {
            cls = c;
            item = b + k;
            return true;
        }
        k -= e - b;
    }
    return false;
}

// One workgroup's tile. XE / ZE: the tile may hold x / z closure rows and face points (false
// only for tiles away from those faces).
template <bool VTI, bool XE, bool ZE>
struct FusedTile {
    static constexpr int NB = VTI ? 3 : 1;
    static constexpr int M66 = VTI ? 1 : 0, M11 = VTI ? 2 : 0;  // coefficient fields c66 and c11b
    static constexpr int CP = FPX * FPZ, PL = 3 * CP;           // LDS words of a component plane, of a ring slot

    const EArgs& __restrict__ A;
    const FusedTiles& FT;
    FusedSmem<VTI>& S;
    float* const ub;  // the ring
    int nx, ny, nz, sx, sy, n3;
    int z0, zo0, zo1, x0, xo0, xo1;
    float ihx, ihy, ihz, ih2x, ih2y, ih2z, ih2x2, ih2y2, ih2z2, rzy;  // (uniform values: in scalar registers)
    D1W dX, dY, dZ;
    // own point
    int lz, lx, ix, iz, cx, cz, col, oi;  // oi: in a component plane
    bool outp, xlo, zlo;
    int xr, xb6, xb8, zr, zb6, zb8;
    float wz[6], tzx;  // tzx: taper factor along z and x
    const float* wx;
    // halo point: role 1 x-halo, 2 z-halo, 3 corner (staging only), 0 none
    int th, role, hrow, hcol, hx, hoff, hi, e0, e1;
    // halo model and ext values of the plane whose fluxes are formed next
    float hm, hl, ve0, ve1, hv[4];

    __device__ __forceinline__ int clx(int x) const { return max(0, min(nx - 1, x)); }
    __device__ __forceinline__ int clz(int z) const { return max(0, min(nz - 1, z)); }
    __device__ __forceinline__ float ld(const float* __restrict__ f, int y, int off) const {
        return gld(f, (unsigned)(max(0, min(ny - 1, y)) * sy + off));
    }
    // Model fields, n3 apart: lam, mu, rho[, c13, eps, c66, c11b]. One base pointer, and n3
    // opaque to the loop-invariant motion (keep_scalars): a pointer per field and component
    // would exceed the scalar registers.
    enum { F_LAM = 0, F_MU = 1, F_C13 = 3, F_EPS = 4, F_C66 = 5, F_C11B = 6 };
    __device__ __forceinline__ const float* mfld(int k) const { return A.lam + k * n3; }
    __device__ __forceinline__ const float* bfld(int m) const { return mfld(m == 0 ? F_MU : (m == 1 ? F_C66 : F_C11B)); }
    __device__ __forceinline__ void keep_scalars() {
        int v = __builtin_amdgcn_readfirstlane(n3);
        asm volatile("" : "+s"(v));
        n3 = v;
        // (and in the bodies near the vector register limit, the addresses formed from these)
        if constexpr (VTI ? (XE || ZE) : (XE && ZE)) asm volatile("" : "+v"(lz), "+v"(lx), "+v"(oi), "+v"(hi), "+v"(zb6), "+v"(zb8));
    }

    __device__ __forceinline__ FusedTile(const EArgs& A_, const FusedTiles& FT_, FusedSmem<VTI>& S_, int tzi, int txi)
        : A(A_), FT(FT_), S(S_), ub(&S_.u[0][0][0][0]), ihx(uniform(1.0f / A_.g.dx)), ihy(uniform(1.0f / A_.g.dy)),
          ihz(uniform(1.0f / A_.g.dz)), dX(ihx), dY(ihy), dZ(ihz) {
        const Geom& g = A.g;
        nx = g.nx; ny = g.ny; nz = g.nz; sx = g.sx; sy = g.sy; n3 = g.n;
        ih2x = uniform(ihx * ihx); ih2y = uniform(ihy * ihy); ih2z = uniform(ihz * ihz);
        ih2x2 = uniform(2.f * ih2x); ih2y2 = uniform(2.f * ih2y); ih2z2 = uniform(2.f * ih2z);
        rzy = uniform(g.dz / g.dy);  // (D_z F_zx has the spacing dy as in the reference)
        fused_tile(nz, FZ, tzi, FT.ntz, z0, zo0, zo1);
        fused_tile(nx, FW, txi, FT.ntx, x0, xo0, xo1);
        const int t = threadIdx.x;
        lz = t & (FZ - 1);
        lx = t >> 5;  // 32 z lanes per x row (a wave holds two x rows)
        ix = x0 + lx;
        iz = z0 + lz;
        cz = min(iz, nz - 1);
        cx = min(ix, nx - 1);
        col = cx * sx + cz;
        oi = (lx + 2) * FPZ + lz + 2;
        outp = ix >= xo0 && ix < xo1 && iz >= zo0 && iz < zo1;
        tzx = gld(A.tz2, cz) * gld(A.tx2, cx);
        // Closure rows along x: two x rows per wave, so the 6 rows at a face fill whole waves
        // and branch uniformly. xr counts rows from the nearer face (0 past the grid, where
        // nothing is output); xb6 / xb8: LDS row of the first of the 6 / 8 points nearest it,
        // in increasing x.
        xlo = ix < nx - 1 - ix;
        xr = !XE ? 8 : (xlo ? ix : max(0, nx - 1 - ix));
        xb8 = max(0, min(FPX - 8, xlo ? 2 - x0 : nx - 6 - x0));
        xb6 = max(0, min(FPX - 6, xlo ? 2 - x0 : nx - 4 - x0));
        wx = S.wd1[xr < 4 ? (xlo ? xr : 4 + xr) : 0];
        // Along z every wave holds closure and interior lanes: all run one code, a window of 6
        // (D1) or 8 (D2) points in increasing z with per-lane weights. Interior lanes put
        // their 5-point stencil (columns lz..lz+4) at the end of the window, which may then
        // start in the preceding row of the plane (weight zero).
        zlo = iz < nz - 1 - iz;
        zr = !ZE ? 8 : (zlo ? iz : max(0, nz - 1 - iz));
        zb6 = zr < 4 ? (zlo ? 2 - z0 : nz - 4 - z0) : lz - 1;
        zb8 = zr < 6 ? (zlo ? 2 - z0 : nz - 6 - z0) : lz - 3;
        if (ZE) {
            const float wi[6] = {0.f, -D1C2, -D1C1, 0.f, D1C1, D1C2};
#pragma unroll
            for (int k = 0; k < 6; k++) wz[k] = ihz * (zr >= 4 ? wi[k] : (zlo ? c_d1w[zr][k] : -c_d1w[zr][5 - k]));
        }
        if (XE || ZE) {
            // values of weight zero at a window's start may come from words not written yet
            float* w = &S.pad[0];
            for (int k = t; k < (int)(sizeof(FusedSmem<VTI>) / sizeof(float)); k += FTHREADS) w[k] = 0.f;
            __syncthreads();
        }
        if (XE && t < 48) {
            const int r = t / 6, k = t % 6;
            S.wd1[r][k] = ihx * (r < 4 ? c_d1w[r][k] : -c_d1w[r - 4][5 - k]);
        }
        // The halo roles go to threads th < 208; th = t except in tiles at the low x face,
        // whose closure rows sit on the first waves: th = t + 256 (mod 512) moves the halo
        // work to the last.
        th = XE && x0 == 0 && xo1 < nx ? (t + 256) & (FTHREADS - 1) : t;
        role = th < 128 ? 1 : (th < 192 ? 2 : (th < 208 ? 3 : 0));
        hrow = hcol = 0;
        hx = ix;
        int hz = iz;
        // e0, e1: the two further points of a halo point's D1 stencil past the staged plane
        // (u_x along x for an x-halo point, u_z along z for a z-halo point)
        e0 = e1 = col;
        if (role == 1) {  // (its z lane is the thread's own)
            const int hr = th >> 5;
            hrow = hr < 2 ? hr : FW + hr;
            hcol = lz + 2;
            hx = x0 - 2 + hrow;
            e0 = clx(hr < 2 ? x0 - 4 + hr : x0 + FW + 2) * sx + cz;
            e1 = clx(hr == 0 ? x0 - 3 : x0 + FW + 3) * sx + cz;
        } else if (role == 2) {
            const int zrw = (th - 128) >> 2, c4 = th & 3;
            hrow = zrw + 2;
            hcol = c4 < 2 ? c4 : FZ + c4;
            hx = x0 + zrw;
            hz = z0 - 2 + hcol;
            e0 = clx(hx) * sx + clz(c4 < 2 ? z0 - 4 + c4 : z0 + FZ + 2) + 2 * n3;
            e1 = clx(hx) * sx + clz(c4 == 0 ? z0 - 3 : z0 + FZ + 3) + 2 * n3;
        } else if (role == 3) {
            const int cr = (th - 192) >> 2, c4 = th & 3;
            hrow = cr < 2 ? cr : FW + cr;
            hcol = c4 < 2 ? c4 : FZ + c4;
            hx = x0 - 2 + hrow;
            hz = z0 - 2 + hcol;
        }
        hoff = clx(hx) * sx + clz(hz);
        hi = hrow * FPZ + hcol;
        hm = hl = ve0 = ve1 = 0.f;
#pragma unroll
        for (int k = 0; k < 4; k++) hv[k] = 0.f;
    }

    // D1 of the closure row of weights w from its 6 points f, f + ldf, ...
    __device__ __forceinline__ float d1xw(const float* w, const float* f, int ldf) const {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < 6; k++) v += w[k] * f[k * ldf];
        return v;
    }
    // D1 at the own z of a plane row f
    __device__ __forceinline__ float d1zw(const float* f) const {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < 6; k++) v += wz[k] * f[zb6 + k];
        return v;
    }
    // D1 at the own point along x (component plane f) and along z
    __device__ __forceinline__ float own_dx(const float* f) const {
        if (XE && xr < 4) return d1xw(wx, f + xb6 * FPZ + lz + 2, FPZ);
        f += oi;
        return dX(f[-2 * FPZ], f[-FPZ], f[FPZ], f[2 * FPZ]);
    }
    __device__ __forceinline__ float own_dz(const float* f) const {
        if (ZE) return d1zw(f + (lx + 2) * FPZ);
        f += oi;
        return dZ(f[-2], f[-1], f[1], f[2]);
    }

    // Stage the own / halo values of a plane into ring slot un.
    __device__ __forceinline__ void stage(float* un, int y, bool halo) const {
#pragma unroll
        for (int c = 0; c < 3; c++) un[c * CP + oi] = ld(A.curr + c * n3, y, col);
        if (halo && role != 0)
#pragma unroll
            for (int c = 0; c < 3; c++) un[c * CP + hi] = ld(A.curr + c * n3, y, hoff);
    }
    __device__ __forceinline__ void load_halo_model(int y) {
        if (role != 1 && role != 2) return;
        hm = ld(mfld(F_MU), y, hoff);
        hl = ld(mfld(F_LAM), y, hoff);
        ve0 = ld(A.curr, y, e0);
        ve1 = ld(A.curr, y, e1);
        if (VTI) {
            hv[0] = ld(mfld(F_C66), y, hoff);
            hv[1] = ld(mfld(F_C11B), y, hoff);
            hv[2] = ld(mfld(F_EPS), y, hoff);
            hv[3] = ld(mfld(F_C13), y, hoff);
        }
    }

    // Stresses and the fluxes differentiated along y at the own point of a plane (u: its
    // ring slot): T_y, F_yx, F_yz (and VTI T_x, T_z; elastic T_x = T_z = T_y).
    __device__ __forceinline__ void stress(const float* u, float dyu1, float mu, float c66, float lam, float eps, float c13,
                                           float& Ty, float& Tx, float& Tz) const {
        const float dxu0 = own_dx(u), dzu2 = own_dz(u + 2 * CP);
        if (!VTI) {
            Ty = Tx = Tz = lam * (dxu0 + dyu1 + dzu2);
        } else {
            const float e2 = 1.f + 2.f * eps;
            const float c11c = e2 * lam, c12 = e2 * (lam + 2.f * mu) - 2.f * c66;
            Ty = c11c * dyu1 + c12 * dxu0 + c13 * dzu2;
            Tx = c11c * dxu0 + c12 * dyu1 + c13 * dzu2;
            Tz = c13 * (dxu0 + dyu1) + lam * dzu2;
        }
    }

    // (A) The D2 coefficient planes and the fluxes differentiated along x and z of a plane
    // (u: its ring slot) into LDS: the own point (coefficients b, stresses Tx, Tz, D_y u_x,
    // D_y u_z) and the thread's halo point (dyh(c): D_y u_c there).
    template <class Dyh>
    __device__ __forceinline__ void flux_plane(const float* u, const float (&b)[NB], float Tx, float Tz, float dyu0,
                                               float dyu2, const Dyh& dyh) {
#pragma unroll
        for (int m = 0; m < NB; m++) S.b[m][lx + 2][lz + 2] = b[m];
        const float mu = b[0];
        S.tx[lx + 2][lz] = Tx;
        S.tz[lx][lz + 2] = Tz;
        S.fxy[lx + 2][lz] = dyu0 * b[M66];
        S.fxz[lx + 2][lz] = own_dz(u) * mu;
        S.fzx[lx][lz + 2] = own_dx(u + 2 * CP) * mu;
        S.fzy[lx][lz + 2] = dyu2 * mu;
        if (role != 1 && role != 2) return;
        S.b[0][hrow][hcol] = hm;
        if (VTI) {
            S.b[M66][hrow][hcol] = hv[0];
            S.b[M11][hrow][hcol] = hv[1];
        }
        const float *h = u + hi, *hw = h + 2 * CP;
        const float dyu1 = dyh(1);
        if (role == 1) {
            // x-halo point: the D1 of u_x along x reaches the ext values
            const int hr = th >> 5;
            const float m2 = hr < 2 ? ve0 : h[-2 * FPZ], m1 = hr == 0 ? ve1 : h[-FPZ];
            const float p1 = hr == 3 ? ve0 : h[FPZ], p2 = hr == 3 ? ve1 : (hr == 2 ? ve0 : h[2 * FPZ]);
            const float dxu0 = dX(m2, m1, p1, p2);
            float dzu2, dzu0;
            if (ZE) {  // (the thread's own z: the same window and weights)
                dzu2 = d1zw(u + 2 * CP + hrow * FPZ);
                dzu0 = d1zw(u + hrow * FPZ);
            } else {
                dzu2 = dZ(hw[-2], hw[-1], hw[1], hw[2]);
                dzu0 = dZ(h[-2], h[-1], h[1], h[2]);
            }
            float T, gxy = hm;
            if (!VTI) {
                T = hl * (dxu0 + dyu1 + dzu2);
            } else {
                const float e2 = 1.f + 2.f * hv[2], c12 = e2 * (hl + 2.f * hm) - 2.f * hv[0];
                T = (e2 * hl) * dxu0 + c12 * dyu1 + hv[3] * dzu2;
                gxy = hv[0];
            }
            S.tx[hrow][lz] = T;
            S.fxy[hrow][lz] = dyh(0) * gxy;
            S.fxz[hrow][lz] = dzu0 * hm;
        } else {
            // z-halo point: the D1 of u_z along z reaches the ext values
            const int zrw = hrow - 2, c4 = th & 3;
            const float m2 = c4 < 2 ? ve0 : hw[-2], m1 = c4 == 0 ? ve1 : hw[-1];
            const float p1 = c4 == 3 ? ve0 : hw[1], p2 = c4 == 3 ? ve1 : (c4 == 2 ? ve0 : hw[2]);
            const float dzu2 = dZ(m2, m1, p1, p2);
            const bool hxlo = hx < nx - 1 - hx;
            const int hxr = hxlo ? hx : max(0, nx - 1 - hx);
            float dxu0, dxu2;
            if (!XE || hxr >= 4) {
                dxu0 = dX(h[-2 * FPZ], h[-FPZ], h[FPZ], h[2 * FPZ]);
                dxu2 = dX(hw[-2 * FPZ], hw[-FPZ], hw[FPZ], hw[2 * FPZ]);
            } else {
                const float* hwx = S.wd1[hxlo ? hxr : 4 + hxr];
                const int hxb = max(0, min(FPX - 6, hxlo ? 2 - x0 : nx - 4 - x0)) * FPZ + hcol;
                dxu0 = d1xw(hwx, u + hxb, FPZ);
                dxu2 = d1xw(hwx, u + 2 * CP + hxb, FPZ);
            }
            float T;
            if (!VTI) T = hl * (dxu0 + dyu1 + dzu2);
            else T = hv[3] * (dxu0 + dyu1) + hl * dzu2;
            S.tz[zrw][hcol] = T;
            S.fzx[zrw][hcol] = dxu2 * hm;
            S.fzy[zrw][hcol] = dyh(2) * hm;
        }
    }

    // D2 coefficients of the own z closure row at plane o.
    __device__ __forceinline__ void load_zrow(int o, float4& t0, float4& t1) const {
        if (ZE && zr < 6) {
            const unsigned e = ((((zlo ? 0 : ny) + o) * nx + cx) * 6 + zr) * 32u;
            t0 = gld4(FT.tab.zc, e);
            t1 = gld4(FT.tab.zc, e + 16);
        }
    }

    // One face's traction SAT at the own point (low or high side of an axis, spacing 1/ih):
    // acc_c -= (sg F_c + K_c S(u_c) ih - imp_c pv_c) / (h H0). F: the stress (normal component
    // cn) and shear fluxes of the point, which hold the terms of the traction that
    // differentiate along the face or carry the normal-stress coefficients; S(u_c): the
    // outward S (times h); K: normal stiffness. tab / e: the point's entry of a face table.
    __device__ __forceinline__ void face_sat(const float4* tab, unsigned e, int bc, bool lo, int cn, float ih, const float (&F)[3],
                                             const float (&K)[3], const float (&su)[3], const float (&pv)[3], float (&acc)[3],
                                             float (&rs)[3]) const {
        const float4 ta = gld4(tab, e);
        const float sg = lo ? -1.f : 1.f, adh = ih * (1.0f / SAT_H0);
#pragma unroll
        for (int c = 0; c < 3; c++) acc[c] -= adh * (sg * F[c] + K[c] * su[c] * ih - (c == cn ? ta.x : ta.y) * pv[c]);
        if (bc == 2) { rs[0] = ta.z; rs[1] = ta.w; rs[2] = gld4(tab, e + 16).x; }
    }

    // (C) The update of plane o (u: its ring slot) at an output point. acc: the terms
    // differentiated along y; b: coefficients of the point; ysat(pv,
    // acc, rs): the SAT of a y face.
    template <class YSat>
    __device__ __forceinline__ void update_plane(const float* u, int o, const float (&b)[NB], float4 tz0,
                                                 float4 tz1, float tfy, float rdt, float (&pv)[3], float (&acc)[3],
                                                 const YSat& ysat) const {
        const unsigned p = (unsigned)(o * sy + ix * sx + iz);
        // D2(b) along x and z of the three components (times h^2); along z the coefficient
        // field is mu for every component
        float d2x[3], d2z[3];
        if (!XE || xr >= 6) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float *f = u + c * CP + oi, *q = &S.b[d2_bfield<VTI>(c, 0)][lx + 2][lz + 2];
                d2x[c] = D2W(q[-2 * FPZ], q[-FPZ], q[0], q[FPZ], q[2 * FPZ])(f[-2 * FPZ], f[-FPZ], f[0], f[FPZ], f[2 * FPZ]);
            }
        } else {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                // (elastic: one coefficient set for the three components)
                const unsigned e = (((((VTI ? 2 * c : 0) + (xlo ? 0 : 1)) * ny + o) * 6 + xr) * nz + iz) * 32u;
                const float4 ta = gld4(FT.tab.xc, e), tb = gld4(FT.tab.xc, e + 16);
                const float* f = u + c * CP + xb8 * FPZ + lz + 2;
                d2x[c] = ta.x * f[0] + ta.y * f[FPZ] + ta.z * f[2 * FPZ] + ta.w * f[3 * FPZ] + tb.x * f[4 * FPZ] +
                         tb.y * f[5 * FPZ] + tb.z * f[6 * FPZ] + tb.w * f[7 * FPZ];
            }
        }
        const float* q = &S.b[0][lx + 2][lz + 2];
        const D2W W(q[-2], q[-1], q[0], q[1], q[2]);
        if (ZE) {
            float w[8] = {0.f, 0.f, 0.f, W.m2, W.m1, W.c0, W.p1, W.p2};
            if (zr < 6) {
                w[0] = tz0.x; w[1] = tz0.y; w[2] = tz0.z; w[3] = tz0.w;
                w[4] = tz1.x; w[5] = tz1.y; w[6] = tz1.z; w[7] = tz1.w;
            }
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float* f = u + c * CP + (lx + 2) * FPZ + zb8;
                float v = w[0] * f[0];
#pragma unroll
                for (int j = 1; j < 8; j++) v += w[j] * f[j];
                d2z[c] = v;
            }
        } else {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float* f = u + c * CP + oi;
                d2z[c] = W(f[-2], f[-1], f[0], f[1], f[2]);
            }
        }
        // outer D1 along x of T / T_x, F_xy, F_xz (components 0, 1, 2), along z of F_zx, F_zy,
        // T / T_z
        const float tf = tzx * tfy;
        const float* PX[3] = {&S.tx[0][lz], &S.fxy[0][lz], &S.fxz[0][lz]};
        const float* PZ[3] = {S.fzx[lx], S.fzy[lx], S.tz[lx]};
#pragma unroll
        for (int c = 0; c < 3; c++) {
            float a = acc[c] + (d2_factor<VTI>(c, 0) == 2.f ? ih2x2 : ih2x) * d2x[c];
            a = a + (d2_factor<VTI>(c, 2) == 2.f ? ih2z2 : ih2z) * d2z[c];
            const float *f = PX[c] + (lx + 2) * FZ, *z = PZ[c] + lz;
            if (!XE || xr >= 4) a = dX.add(a, f[-2 * FZ], f[-FZ], f[FZ], f[2 * FZ]);
            else a = a + d1xw(wx, PX[c] + xb6 * FZ, FZ);
            if (ZE) a = a + (c == 0 ? d1zw(PZ[c]) * rzy : d1zw(PZ[c]));
            else if (c == 0) a = dY.add(a, z[0], z[1], z[3], z[4]);  // (spacing dy)
            else a = dZ.add(a, z[0], z[1], z[3], z[4]);
            acc[c] = a;
            if (A.prev_tapered) pv[c] *= tf;
        }
        float rs[3] = {1.f, 1.f, 1.f};
        if (ZE && zr == 0) {
            const int bc = zlo ? A.bc[0] : A.bc[1], st = zlo ? 1 : -1;
            if (bc == 1 || bc == 2) {
                float su[3];
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const float* f = u + c * CP + oi;
                    su[c] = c_sat_s[0] * f[0] + c_sat_s[1] * f[st] + c_sat_s[2] * f[2 * st] + c_sat_s[3] * f[3 * st];
                }
                face_sat(FT.tab.zf, (((zlo ? 0 : ny) + o) * nx + ix) * 32u, bc, zlo, 2, ihz,
                         {S.fzx[lx][lz + 2], S.fzy[lx][lz + 2], S.tz[lx][lz + 2]}, {b[0], b[0], 2.f * b[0]}, su, pv, acc, rs);
            }
        }
        if (XE && xr == 0) {
            const int bc = xlo ? A.bc[2] : A.bc[3], st = xlo ? FPZ : -FPZ;
            if (bc == 1 || bc == 2) {
                float su[3];
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const float* f = u + c * CP + oi;
                    su[c] = c_sat_s[0] * f[0] + c_sat_s[1] * f[st] + c_sat_s[2] * f[2 * st] + c_sat_s[3] * f[3 * st];
                }
                face_sat(FT.tab.xf, (((xlo ? 0 : ny) + o) * nz + iz) * 32u, bc, xlo, 0, ihx,
                         {S.tx[lx + 2][lz], S.fxy[lx + 2][lz], S.fxz[lx + 2][lz]}, {VTI ? b[M11] : 2.f * b[0], b[M66], b[0]}, su, pv, acc, rs);
            }
        }
        ysat(pv, acc, rs);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            float nv = acc[c] * rdt + (2.f * u[c * CP + oi] - pv[c]);
            nv *= rs[c];
            gst(A.next, c * n3 + p, nv * tf);
        }
    }

    // ---- planes [ya, yb) inside [6, ny-6), marching along y
    __device__ __forceinline__ void march(int ya, int yb) {
        // state carried along y
        float qb[NB][6];                // D2 coefficient fields at o-2..o+3
        float tq[5], fyxq[5], fyzq[5];  // T_y, F_yx, F_yz at o-2..o+2
        float txq[2], tzq[2];           // VTI: T_x, T_z at o+1, o+2
        float yp[3] = {0.f, 0.f, 0.f};  // elastic: D2 pairs of mu along y: p1 from o-1, p2 from o-1, o-2
        float uy3, uy4;                 // u_y at o+3, o+4
        const float* __restrict__ curr = A.curr;
        const int o0 = ya - 4;
        // (the coefficient planes before o0+2 = ya-2 are not read)
#pragma unroll
        for (int k = 0; k < 5; k++) {
#pragma unroll
            for (int m = 0; m < NB; m++) qb[m][k] = k < 4 ? 0.f : ld(bfld(m), o0 + 2, col);
            tq[k] = fyxq[k] = fyzq[k] = 0.f;
        }
#pragma unroll
        for (int k = 0; k < 2; k++) txq[k] = tzq[k] = 0.f;
        uy3 = ld(curr + n3, o0 + 3, col);
        int so = o0 % FRING;  // slot of plane o (o0 >= 2)
        auto slot = [&](int k) { const int s = so + k; return ub + (s >= FRING ? s - FRING : (s < 0 ? s + FRING : s)) * PL; };
        // the look-ahead of the first iteration reads plane o0+2 and u_y at planes o0, o0+1 of
        // the own column
        slot(0)[CP + oi] = ld(curr + n3, o0, col);
        slot(1)[CP + oi] = ld(curr + n3, o0 + 1, col);
        stage(slot(2), o0 + 2, true);
        __syncthreads();

        // Iteration o: (A) fluxes of plane o into LDS, plane o+3 into the ring; barrier; (C)
        // the look-ahead fluxes of plane o+2 and the update of plane o; barrier.
        for (int o = o0; o < yb; o++) {
            keep_scalars();
            const bool live = o >= ya;
            // plane o+3, staged at the end of (A)
            const float nux = ld(curr, o + 3, col), nuz = ld(curr + 2 * n3, o + 3, col);
            uy4 = ld(curr + n3, o + 4, col);
#pragma unroll
            for (int m = 0; m < NB; m++) qb[m][5] = ld(bfld(m), o + 3, col);
            float nh[3] = {0.f, 0.f, 0.f};
            if (role != 0)
#pragma unroll
                for (int c = 0; c < 3; c++) nh[c] = ld(curr + c * n3, o + 3, hoff);
            // loads used in (C)
            const float lam2 = ld(mfld(F_LAM), o + 2, col);
            float eps2 = 0.f, c132 = 0.f;
            if (VTI) {
                eps2 = ld(mfld(F_EPS), o + 2, col);
                c132 = ld(mfld(F_C13), o + 2, col);
            }
            float tfy = 0.f, rdt = 0.f, pv[3] = {0.f, 0.f, 0.f}, acc[3] = {0.f, 0.f, 0.f};
            if (live) {
                tfy = gld(A.ty2, o);
                rdt = ld(FT.rdt, o, col);
#pragma unroll
                for (int c = 0; c < 3; c++) pv[c] = ld(A.prev + c * n3, o, col);
            }
            // elastic: the y pairs of mu from plane o (its neighbours' are carried along)
            float py1 = 0.f, py2 = 0.f;
            if (!VTI) {
                py1 = d2_pair1(qb[0][1], qb[0][2], qb[0][3], qb[0][4]);
                py2 = d2_pair2(qb[0][2], qb[0][3], qb[0][4]);
            }
            const float* const uo = slot(0);
            float bo[NB];
#pragma unroll
            for (int m = 0; m < NB; m++) bo[m] = qb[m][2];
            if (live) {
                const float *um2 = slot(-2), *um1 = slot(-1), *up1 = slot(1), *up2 = slot(2);
                float dy[3];
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const int q = c * CP + oi, m = d2_bfield<VTI>(c, 1);
                    const float vm2 = um2[q], vm1 = um1[q], v0 = uo[q], vp1 = up1[q], vp2 = up2[q];
                    const D2W W = VTI ? D2W(qb[m][0], qb[m][1], qb[m][2], qb[m][3], qb[m][4]) : D2W(yp[2], yp[0], py1, py2);
                    acc[c] = (d2_factor<VTI>(c, 1) == 2.f ? ih2y2 : ih2y) * W(vm2, vm1, v0, vp1, vp2);
                    dy[c] = dY(vm2, vm1, vp1, vp2);  // (of u_x and u_z)
                }
                // (the look-ahead of this iteration has not run yet: the queues end at o+1)
                flux_plane(uo, bo, VTI ? txq[0] : tq[3], VTI ? tzq[0] : tq[3], dy[0], dy[2],
                           [&](int c) { const int q = c * CP + hi; return dY(um2[q], um1[q], up1[q], up2[q]); });
            }
            {
                // (the slot held plane o-3, last read in iteration o-1)
                float* const un = slot(3);
                un[oi] = nux;
                un[CP + oi] = uy3;
                un[2 * CP + oi] = nuz;
                if (role != 0)
#pragma unroll
                    for (int c = 0; c < 3; c++) un[c * CP + hi] = nh[c];
            }
            if (live) __syncthreads();

            float4 tz0{}, tz1{};
            if (live) load_zrow(o, tz0, tz1);
            {
                const float* const u2 = slot(2);
                float Ty, Tx, Tz;
                stress(u2, dY(uo[CP + oi], slot(1)[CP + oi], uy3, uy4), qb[0][4], qb[M66][4], lam2, eps2, c132, Ty, Tx, Tz);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    tq[k] = tq[k + 1]; fyxq[k] = fyxq[k + 1]; fyzq[k] = fyzq[k + 1];
                }
                tq[4] = Ty;
                fyxq[4] = own_dx(u2 + CP) * qb[M66][4];
                fyzq[4] = own_dz(u2 + CP) * qb[0][4];
                if (VTI) {
                    txq[0] = txq[1]; txq[1] = Tx;
                    tzq[0] = tzq[1]; tzq[1] = Tz;
                }
            }
            if (live && outp) {
                acc[0] = dY.add(acc[0], fyxq[0], fyxq[1], fyxq[3], fyxq[4]);
                acc[1] = dY.add(acc[1], tq[0], tq[1], tq[3], tq[4]);
                acc[2] = dY.add(acc[2], fyzq[0], fyzq[1], fyzq[3], fyzq[4]);
                update_plane(uo, o, bo, tz0, tz1, tfy, rdt, pv, acc,
                             [](const float (&)[3], float (&)[3], float (&)[3]) {});
            }
            if (o + 1 >= ya) load_halo_model(o + 1);
            uy3 = uy4;
            yp[2] = yp[1];
            yp[1] = py2;
            yp[0] = py1;
#pragma unroll
            for (int k = 0; k < 5; k++)
#pragma unroll
                for (int m = 0; m < NB; m++) qb[m][k] = qb[m][k + 1];
            so = so + 1 == FRING ? 0 : so + 1;
            __syncthreads();
        }
    }

    // ---- rows r0..r0+2 (r0 = 0 or 3) of the 6 planes at a y face. Planes are counted from
    // the face, j = 0..9: the closure rows j < 6 read planes 0..7 of u and of the fluxes T_y,
    // F_yx, F_yz, whose D1 reads u_y to plane 9. Planes 6 and 7 pass through two ring slots
    // first; planes 0..5 then fill the ring for the rows. The weights of a row come from
    // constant tables by its uniform index (a dense row: rows 4 and 5 of D1 are its interior
    // stencil). Three rows per workgroup: six would take 9 more registers and twice the time,
    // which on small grids is the step's.
    __device__ __forceinline__ void yface(bool hi_face, int r0) {
        const float* __restrict__ curr = A.curr;
        const float sg = hi_face ? -ihy : ihy;  // D1 changes sign at the high face
        auto Y = [&](int j) { return hi_face ? ny - 1 - j : j; };
        // own column beyond the ring: u_x, u_z of planes 6, 7; u_y of planes 4..9
        float ux[2], uz[2], uy[6], hh[2][3];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            ux[k] = ld(curr, Y(6 + k), col);
            uz[k] = ld(curr + 2 * n3, Y(6 + k), col);
#pragma unroll
            for (int c = 0; c < 3; c++) hh[k][c] = role != 0 ? ld(curr + c * n3, Y(6 + k), hoff) : 0.f;
        }
#pragma unroll
        for (int k = 0; k < 6; k++) uy[k] = ld(curr + n3, Y(4 + k), col);
        float accy[3][3];  // D1 along y of F_yx, T_y, F_yz at rows r0..r0+2
#pragma unroll
        for (int r = 0; r < 3; r++) accy[r][0] = accy[r][1] = accy[r][2] = 0.f;
        float f0[3] = {0.f, 0.f, 0.f};  // F_yx, T_y, F_yz of the face plane
        float mu, c66, lam, eps = 0.f, c13 = 0.f;  // model of the plane whose fluxes are formed next
        auto model = [&](int j) {
            keep_scalars();
            const int y = Y(j);
            mu = ld(mfld(F_MU), y, col);
            c66 = VTI ? ld(mfld(F_C66), y, col) : mu;
            lam = ld(mfld(F_LAM), y, col);
            if (VTI) {
                eps = ld(mfld(F_EPS), y, col);
                c13 = ld(mfld(F_C13), y, col);
            }
        };
        auto ahead = [&](int j, int jn, const float* u, float dyu1) {  // jn: the plane after this one
            float F[3], Tx, Tz;
            const float m = mu, g = c66;
            stress(u, dyu1, mu, c66, lam, eps, c13, F[1], Tx, Tz);
            model(jn);
            F[0] = own_dx(u + CP) * g;
            F[2] = own_dz(u + CP) * m;
#pragma unroll
            for (int r = 0; r < 3; r++) {
                const float w = c_y1w[r0 + r][j] * sg;
#pragma unroll
                for (int c = 0; c < 3; c++) accy[r][c] += w * F[c];
            }
            if (j == 0) { f0[0] = F[0]; f0[1] = F[1]; f0[2] = F[2]; }
        };
        if (r0 != 0) {
            model(6);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                float* const un = ub + k * PL;
                un[oi] = ux[k];
                un[CP + oi] = uy[2 + k];
                un[2 * CP + oi] = uz[k];
                if (role != 0)
#pragma unroll
                    for (int c = 0; c < 3; c++) un[c * CP + hi] = hh[k][c];
            }
            __syncthreads();
            ahead(6, 7, ub, sg * (D1C1 * (uy[3] - uy[1]) + D1C2 * (uy[4] - uy[0])));
            ahead(7, 0, ub + PL, sg * (D1C1 * (uy[4] - uy[2]) + D1C2 * (uy[5] - uy[1])));
            __syncthreads();
        } else {
            model(0);
        }
#pragma unroll 2
        for (int j = 0; j < 6; j++) stage(ub + j * PL, Y(j), true);
        load_halo_model(Y(r0));
        __syncthreads();
        // D1 along y of component c at row j of the column at q of a component plane; v6, v7:
        // its values at planes 6, 7
        auto dy = [&](int j, int c, int q, float v6, float v7) {
            float v = c_y1w[j][6] * v6 + c_y1w[j][7] * v7;
#pragma unroll
            for (int k = 0; k < 6; k++) v += c_y1w[j][k] * ub[k * PL + c * CP + q];
            return v * sg;
        };
        // planes 0..4 for rows 0..2; 0 and 2..7 for rows 3..5
        const int step0 = r0 == 0 ? 1 : 2, last = r0 == 0 ? 4 : 5;
#pragma unroll 1
        for (int j = 0; j <= last;) {
            const int jn = j == 0 ? step0 : j + 1;
            ahead(j, min(jn, last), ub + j * PL, dy(j, 1, oi, uy[2], uy[3]));
            j = jn;
        }

#pragma unroll 1
        for (int r = r0; r < r0 + 3; r++) {
            keep_scalars();
            const int o = Y(r);
            const float* const u = ub + r * PL;
            model(r);
            float bo[NB];
#pragma unroll
            for (int m = 0; m < NB; m++) bo[m] = ld(bfld(m), o, col);
            float acc[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                // (elastic: one coefficient set for the three components)
                const unsigned e = ((((VTI ? 2 * c : 0) + (hi_face ? 1 : 0)) * 6 + r) * nx + cx) * nz + cz;
                const float4 ta = gld4(FT.tab.yc, e * 32u), tb = gld4(FT.tab.yc, e * 32u + 16);
                const float v6 = c == 0 ? ux[0] : (c == 1 ? uy[2] : uz[0]), v7 = c == 0 ? ux[1] : (c == 1 ? uy[3] : uz[1]);
                const float* f = ub + c * CP + oi;
                const float v = ta.x * f[0] + ta.y * f[PL] + ta.z * f[2 * PL] + ta.w * f[3 * PL] + tb.x * f[4 * PL] +
                                tb.y * f[5 * PL] + tb.z * v6 + tb.w * v7;
                acc[c] = (d2_factor<VTI>(c, 1) == 2.f ? ih2y2 : ih2y) * v + accy[0][c];
            }
            float Ty, Tx, Tz;
            stress(u, dy(r, 1, oi, uy[2], uy[3]), mu, c66, lam, eps, c13, Ty, Tx, Tz);
            flux_plane(u, bo, Tx, Tz, dy(r, 0, oi, ux[0], ux[1]), dy(r, 2, oi, uz[0], uz[1]),
                       [&](int c) { return dy(r, c, hi, hh[0][c], hh[1][c]); });
            const float tfy = gld(A.ty2, o), rdt = ld(FT.rdt, o, col);
            float pv[3];
#pragma unroll
            for (int c = 0; c < 3; c++) pv[c] = ld(A.prev + c * n3, o, col);
            float4 tz0{}, tz1{};
            load_zrow(o, tz0, tz1);
            __syncthreads();
            if (outp)
                update_plane(u, o, bo, tz0, tz1, tfy, rdt, pv, acc,
                             [&](const float (&p)[3], float (&a)[3], float (&rs)[3]) {
                                 const int bc = hi_face ? A.bc[5] : A.bc[4];
                                 if (r != 0 || (bc != 1 && bc != 2)) return;
                                 float su[3];
#pragma unroll
                                 for (int c = 0; c < 3; c++) {
                                     const float* f = ub + c * CP + oi;
                                     su[c] = c_sat_s[0] * f[0] + c_sat_s[1] * f[PL] + c_sat_s[2] * f[2 * PL] + c_sat_s[3] * f[3 * PL];
                                 }
                                 face_sat(FT.tab.yf, (((hi_face ? nx : 0) + ix) * nz + iz) * 32u, bc, !hi_face, 1, ihy, f0,
                                          {bo[M66], VTI ? bo[M11] : 2.f * bo[0], bo[0]}, su, p, a, rs);
                             });
#pragma unroll
            for (int c = 0; c < 3; c++) {
                accy[0][c] = accy[1][c];
                accy[1][c] = accy[2][c];
            }
            if (r < r0 + 2) load_halo_model(Y(r + 1));
            __syncthreads();
        }
    }
};

}  // namespace fwi3d
