// Time-invariant boundary data of the fused elastic / VTI step (fused.hpp), formed once
// per propagation from the converted model:
//
//   D2 closure coefficients  c_j = sum_k w_rjk b_k of the 6 rows at each face: a
//                            closure row then is sum_j c_j u_j, 8 products, the same code
//                            for every row (w_rjk: kD2Closure; b: the coefficient field of
//                            the component along that axis).
//   face values              impedances over dt of the absorbing traction SATs and the
//                            reciprocals of their implicit scaling (e_scale), at every
//                            point of the six faces.
//
// An edge tile of the step reads them for its closure rows and face points only. Without
// them a closure row needs its 8 coefficient values and row-specific code (~22 products per
// coefficient field, one branch per row), and a face point five square roots and three
// divisions per step.
#pragma once
#include "elastic.hpp"

namespace fwi3d {

// Device pointers of one shot's tables; each entry is two float4.
//   zc[((face ny + y) nx + x) 6 + row], mu; 8 coefficients in increasing z
//   xc[((2 set + face) ny + y) 6 + row) nz + z]; sets: VTI c11b, c66, mu (the components
//      x, y, z), elastic mu only; 8 coefficients in increasing x
//   yc[((2 set + face) 6 + row) nx + x) nz + z]; sets: VTI c66, c11b, mu (the components x,
//      y, z), elastic mu only; 8 coefficients counted from the face
//   zf[(face ny + y) nx + x], xf[(face ny + y) nz + z], yf[(face nx + x) nz + z]:
//      {P impedance / dt, S impedance / dt, 1 / scale of u_x, u_y}, {of u_z, -, -, -}
//      (impedances zero unless the face absorbs)
struct ClosureTabs {
    const float4* zc;
    const float4* xc;
    const float4* yc;
    const float4* zf;
    const float4* xf;
    const float4* yf;
};

// float4 entries of the tables, in the order of their one allocation.
struct ClosureSizes {
    size_t zc, xc, yc, zf, xf, yf;
    __host__ __device__ size_t total() const { return zc + xc + yc + zf + xf + yf; }
};
inline ClosureSizes closure_sizes(bool vti, const Geom& g) {
    const size_t nx = g.nx, ny = g.ny, nz = g.nz, sets = vti ? 3 : 1;
    return ClosureSizes{24 * ny * nx, 24 * sets * ny * nz, 24 * sets * nx * nz, 4 * ny * nx, 4 * ny * nz, 4 * nx * nz};
}
inline ClosureTabs closure_tabs(float4* base, const ClosureSizes& s) {
    ClosureTabs t;
    t.zc = base;
    t.xc = t.zc + s.zc;
    t.yc = t.xc + s.xc;
    t.zf = t.yc + s.yc;
    t.xf = t.zf + s.zf;
    t.yf = t.xf + s.xf;
    return t;
}

__host__ __device__ constexpr bool d2_uses(int r, int j) {
    for (int e = 0; e < 132; e++)
        if (kD2Closure[e].r == r && kD2Closure[e].j == j) return true;
    return false;
}
// c_j of row R: the non-zero w_Rjk b_k in increasing k.
template <int R, int J, int E>
__device__ __forceinline__ float d2_cj(float acc, const float (&b)[8]) {
    if constexpr (E == 132) return acc;
    else if constexpr (kD2Closure[E].r == R && kD2Closure[E].j == J)
        return d2_cj<R, J, E + 1>(acc + D2Term<E>::w * b[kD2Closure[E].k], b);
    else return d2_cj<R, J, E + 1>(acc, b);
}
template <int R, int J>
__device__ __forceinline__ void d2_coef_row(const float (&b)[8], float (&c)[8]) {
    if constexpr (J < 8) {
        if constexpr (d2_uses(R, J)) c[J] = d2_cj<R, J, 0>(-0.0f, b);
        else c[J] = 0.f;
        d2_coef_row<R, J + 1>(b, c);
    }
}
__device__ __forceinline__ void d2_coefs(int r, const float (&b)[8], float (&c)[8]) {
    switch (r) {
        case 0: d2_coef_row<0, 0>(b, c); break;
        case 1: d2_coef_row<1, 0>(b, c); break;
        case 2: d2_coef_row<2, 0>(b, c); break;
        case 3: d2_coef_row<3, 0>(b, c); break;
        case 4: d2_coef_row<4, 0>(b, c); break;
        default: d2_coef_row<5, 0>(b, c); break;
    }
}

// dt^2 / rho, the factor of the acceleration in the update (padding: zero).
__global__ __launch_bounds__(256) void rdt_field(float* __restrict__ out, const float* __restrict__ rho, float dt2, Geom g) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < g.n) out[i] = (int)(i % g.pz) < g.nz ? dt2 / rho[i] : 0.f;
}

// One thread per table entry (grid-stride over the entries of all tables).
template <bool VTI>
__global__ __launch_bounds__(256) void closure_tables(EArgs A, float4* __restrict__ base, ClosureSizes S) {
    const Geom g = A.g;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const long long nzc = (long long)S.zc / 2, nxc = (long long)S.xc / 2, nyc = (long long)S.yc / 2, nzf = (long long)S.zf / 2,
                    nxf = (long long)S.xf / 2, nyf = (long long)S.yf / 2;
    const long long nc = nzc + nxc + nyc, n = nc + nzf + nxf + nyf;
    const ECoef<VTI> M{A.lam, A.mu, A.rho, A.c13, A.eps, A.c66};
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x) {
        float4* out = base + 2 * e;
        if (e < nc) {
            const int ax = e < nzc ? 2 : (e < nzc + nxc ? 0 : 1);
            int q = (int)(e - (ax == 2 ? 0 : (ax == 0 ? nzc : nzc + nxc))), r, p0, set = 0, hi;
            if (ax == 2) {
                r = q % 6;
                q /= 6;
                p0 = g.at(q % nx, (q / nx) % ny, 0);
                hi = q / (nx * ny);
            } else {
                const int z = q % nz;
                q /= nz;
                int x = 0, y = 0;
                if (ax == 1) {
                    x = q % nx;
                    q /= nx;
                }
                r = q % 6;
                q /= 6;
                if (ax == 0) {
                    y = q % ny;
                    q /= ny;
                }
                p0 = g.at(x, y, z);
                hi = q & 1;
                set = q >> 1;
            }
            const int st = ax_stride(g, ax), len = ax_len(g, ax);
            const int m = VTI && ax != 2 ? d2_bfield<VTI>(set, ax) : 0;
            const float* f = m == 2 ? A.c11b : (m == 1 ? A.c66 : A.mu);
            const bool flip = hi && ax != 1;
            float b[8], c[8];
#pragma unroll
            for (int k = 0; k < 8; k++) b[k] = gld(f, p0 + (hi ? len - 1 - k : k) * st);
            d2_coefs(r, b, c);
            out[0] = flip ? make_float4(c[7], c[6], c[5], c[4]) : make_float4(c[0], c[1], c[2], c[3]);
            out[1] = flip ? make_float4(c[3], c[2], c[1], c[0]) : make_float4(c[4], c[5], c[6], c[7]);
            continue;
        }
        long long q = e - nc;
        int ix, iy, iz, ax, hi;
        if (q < nzf) {
            ax = 2; ix = (int)(q % nx); iy = (int)(q / nx % ny); hi = (int)(q / nx / ny); iz = hi ? nz - 1 : 0;
        } else if ((q -= nzf) < nxf) {
            ax = 0; iz = (int)(q % nz); iy = (int)(q / nz % ny); hi = (int)(q / nz / ny); ix = hi ? nx - 1 : 0;
        } else {
            q -= nxf;
            ax = 1; iz = (int)(q % nz); ix = (int)(q / nz % nx); hi = (int)(q / nz / nx); iy = hi ? ny - 1 : 0;
        }
        const int p = g.at(ix, iy, iz);
        const bool ab = A.bc[ax == 2 ? hi : (ax == 0 ? 2 + hi : 4 + hi)] == 2;
        out[0] = make_float4(ab ? M.pimp(ax, p) / A.dt : 0.f, ab ? 0.5f * sqrtf(M.mu[p] * M.rho[p]) / A.dt : 0.f,
                             1.f / e_scale<VTI>(g, A.bc, M, p, ix, iy, iz, 0, A.dt),
                             1.f / e_scale<VTI>(g, A.bc, M, p, ix, iy, iz, 1, A.dt));
        out[1] = make_float4(1.f / e_scale<VTI>(g, A.bc, M, p, ix, iy, iz, 2, A.dt), 0.f, 0.f, 0.f);
    }
}

}  // namespace fwi3d
