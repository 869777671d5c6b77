// Gradient vector flow by the full-multigrid (FMG) solver.
//
// Per component c, `iterations` defect-correction steps are run on the
// linear system  mu*lap(v) - |F|^2 v = -|F|^2 F_c  (mirror boundary):
//   r = fmgResidual(f);  e = FMG(r);  f += e
// (runFMGGVF, gradientVectorFlow.cpp:729-1005).  FMG recurses over
// levels+1 cubic grids (calculateNewSize: next power of two of the largest
// extent, halved), each smoothed by red-black Gauss-Seidel sweeps.  All grid
// buffers are allocated once per call (the reference allocates a fresh image
// per helper call) and the restricted |F|^2 pyramid is built once, since it
// does not change between cycles.  Arithmetic is float in the reference's
// operation order; the smoother divides with an IEEE division where the
// reference uses native_divide.
//
// Layout: every grid is kept as two arrays, its red cells (x + y + z even)
// and its black ones, rows padded to four elements.  A half-sweep then reads
// the other colour, r and s of its own and writes its own: half the bytes of
// whole grids, every lane at work, in place.  The mirror of a boundary cell
// (0 -> 2, N-1 -> N-3) has the cell's colour, so the boundary cells are
// stored by the thread that computes their mirror.  A red half-sweep does not
// read red cells, so what precedes one (zeroing, prolongation) is part of it;
// the last half-sweep of a cycle adds to f, and both residuals are restricted
// as they are made.
//
// The components do not depend on each other: grids up to 2^22 cells run all
// three in one launch (a half-sweep of 64^3 cells takes 3 us for one and for
// three), larger ones a component at a time, so that a phase's r, v and s
// (201 MB at 256^3) can stay in the last-level cache.  Grids above 2^27 cells
// keep one component's buffers only and run the cycles one after another, as
// do smaller ones in a workspace that holds no more.
//
// 256^3, two levels, 10 cycles: 27.7 ms on whole grids, 15.1 ms split,
// 13.1 ms with the zeroing, prolongation, restriction and f += e passes gone
// into their neighbours.  Bound by the bytes of the finest grid (the
// half-sweeps 24-28 us for 134 MB; two of them to a launch would have to read
// the halo of both).
#include <math.h>

#include <algorithm>
#include <vector>

#include "tsf_common.hpp"

namespace tsf {

// One grid: extents, elements per row and colour, cells per colour.
struct Grid {
    Dims d;
    int xs;
    i64 m;
    explicit Grid(Dims e) : d(e), xs((((e.X + 1) / 2) + 3) & ~3), m((i64)xs * e.Y * e.Z) {}
    __host__ __device__ i64 row(int y, int z) const { return (i64)xs * ((i64)y + (i64)d.Y * z); }
};
// A colour-split array is its red cells followed by its black ones.
struct Trio {
    float* p[3];
};

__device__ __forceinline__ void ld4(float (&v)[4], const float* p) { __builtin_memcpy(v, p, 16); }
__device__ __forceinline__ void ld4a(float (&v)[4], const float* p) {
    const float4 q = *reinterpret_cast<const float4*>(p);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
}
__device__ __forceinline__ void st4a(float* p, const float (&v)[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
// the array that holds the even (odd) x of a row: red cells have x + y + z even
__device__ __forceinline__ const float* even_x(const Grid& g, const float* a, int y, int z) {
    return a + g.row(y, z) + (((y + z) & 1) ? g.m : 0);
}
__device__ __forceinline__ const float* odd_x(const Grid& g, const float* a, int y, int z) {
    return a + g.row(y, z) + (((y + z) & 1) ? 0 : g.m);
}
// thread -> quad i (elements i .. i + 3 of a row of each colour) and row y
__device__ __forceinline__ bool quad_of(int xs, int rows, int& i, int& y) {
    const int q = xs >> 2, t = (int)(blockIdx.x * 256 + threadIdx.x);
    y = t / q;
    i = 4 * (t - y * q);
    return y < rows;
}
static dim3 quad_grid(int xs, int rows, int planes, int comps) {
    return dim3((unsigned)(((i64)(xs >> 2) * rows + 255) / 256), (unsigned)planes, (unsigned)comps);
}

// s = |F|^2
__global__ void __launch_bounds__(256) k_sqrmag(const float* __restrict__ fx, const float* __restrict__ fy,
                                                const float* __restrict__ fz, Grid g, float* __restrict__ s) {
    int i, y;
    if (!quad_of(g.xs, g.d.Y, i, y)) return;
    const int z = blockIdx.y;
    const int odd = (y + z) & 1;
    float e[2][4], a[8], b[8], c[8];
    const i64 q = g.d.at(2 * i, y, z);
    if (2 * i + 7 < g.d.X) {
        __builtin_memcpy(a, fx + q, 32);
        __builtin_memcpy(b, fy + q, 32);
        __builtin_memcpy(c, fz + q, 32);
    } else {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const bool in = 2 * i + j < g.d.X;
            a[j] = in ? fx[q + j] : 0.0f;
            b[j] = in ? fy[q + j] : 0.0f;
            c[j] = in ? fz[q + j] : 0.0f;
        }
    }
#pragma unroll
    for (int j = 0; j < 8; j++) e[j & 1][j >> 1] = a[j] * a[j] + b[j] * b[j] + c[j] * c[j];
    float* o = s + g.row(y, z) + i;
    st4a(o + (odd ? g.m : 0), e[0]);
    st4a(o + (odd ? 0 : g.m), e[1]);
}

// fmgResidual, kernels_no_3d_write.cl:2303-2348 (finest grid, h = 1); F_c and
// f are plain arrays, |F|^2 comes from s.  Rows past X get zeros.
__device__ __forceinline__ float fmg_residual_of(float fc, float c, float sq, float nb, float mu) {
    const float residue = mu * (nb - 6.0f * c);
    return -sq * fc - (residue - sq * c);
}
// the residuals x = 2 i .. 2 i + 7 of row (y, z), also stored in r
__device__ __forceinline__ void fmg_residual_row(const float* __restrict__ Fc, const float* __restrict__ f,
                                                 const float* __restrict__ s, const Grid& g, float mu, int y, int z,
                                                 int i, float* __restrict__ r, float* ev, float* od) {
    const int X = g.d.X;
    const int py = remap(y, g.d.Y), pz = remap(z, g.d.Z);
    const i64 sy = X, sz = (i64)X * g.d.Y, q = g.d.at(2 * i, py, pz);  // rows py, pz are interior: q - 1 .. q + 8 exist
    float e[2][4];
    if (2 * i + 7 < X) {
        float c[10], yp[8], ym[8], zp[8], zm[8], fc[8], se[4], so[4];
        __builtin_memcpy(c + 1, f + q, 32);
        c[0] = f[q - 1];
        c[9] = f[q + 8];
        __builtin_memcpy(yp, f + q + sy, 32);
        __builtin_memcpy(ym, f + q - sy, 32);
        __builtin_memcpy(zp, f + q + sz, 32);
        __builtin_memcpy(zm, f + q - sz, 32);
        __builtin_memcpy(fc, Fc + q, 32);
        ld4a(se, even_x(g, s, py, pz) + i);
        ld4a(so, odd_x(g, s, py, pz) + i);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            float nb = c[j + 2];
            nb = nb + c[j];
            nb = nb + yp[j];
            nb = nb + ym[j];
            nb = nb + zp[j];
            nb = nb + zm[j];
            e[j & 1][j >> 1] = fmg_residual_of(fc[j], c[j + 1], (j & 1) ? so[j >> 1] : se[j >> 1], nb, mu);
        }
        if (i == 0) e[0][0] = e[0][1];
        if (2 * i + 7 == X - 1) e[1][3] = e[1][2];
    } else {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            float v = 0.0f;
            if (2 * i + j < X) {
                const int x = remap(2 * i + j, X);
                const i64 k = g.d.at(x, py, pz);
                float nb = f[k + 1];
                nb = nb + f[k - 1];
                nb = nb + f[k + sy];
                nb = nb + f[k - sy];
                nb = nb + f[k + sz];
                nb = nb + f[k - sz];
                const float* sr = (x & 1) ? odd_x(g, s, py, pz) : even_x(g, s, py, pz);
                v = fmg_residual_of(Fc[k], f[k], sr[x >> 1], nb, mu);
            }
            e[j & 1][j >> 1] = v;
        }
    }
    const int odd = (y + z) & 1;
    float* o = r + g.row(y, z) + i;
    st4a(o + (odd ? g.m : 0), e[0]);
    st4a(o + (odd ? 0 : g.m), e[1]);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        ev[j] = e[0][j];
        od[j] = e[1][j];
    }
}
__global__ void __launch_bounds__(256) k_fmg_residual(const float* __restrict__ Fc, const float* __restrict__ f,
                                                      const float* __restrict__ s, Grid g, float mu,
                                                      float* __restrict__ r) {
    int i, y;
    float ev[4], od[4];
    if (quad_of(g.xs, g.d.Y, i, y)) fmg_residual_row(Fc, f, s, g, mu, y, blockIdx.y, i, r, ev, od);
}

// GVFgaussSeidel / GVFgaussSeidel2 (the half-sweeps), kernels_no_3d_write.cl:
// 2071-2150: the cells of colour BLACK from the other colour.
__device__ __forceinline__ float gs_value(float nb, float r, float s, float mu, float h) {
    const float num = 2.0f * mu * nb - 2.0f * h * h * r;
    const float den = 12.0f * mu + h * h * s;
    return num / den;
}
// Where a red half-sweep takes the black cells from: the grid, the injected
// coarse grid (prolongate2, kernels_no_3d_write.cl:2248-2266), the grid plus
// that (prolongate), or nowhere (zeros).
enum { FROM_GRID, FROM_COARSE, FROM_SUM, FROM_ZERO };
struct HalfArgs {
    Trio v, r;
    const float* s;
    Grid g;
    float mu, h;
    int zc;
    Trio c;  // FROM_COARSE, FROM_SUM: the coarse grid
    Grid cg;
    Trio f;  // ADD: plain arrays
};
template <int FROM>
struct Other {
    const float* o;  // the other colour's cells
    const float* c;
    const HalfArgs& a;
    // four elements from i (a multiple of 4) / element i of row (y, z); i = -1
    // and i = the row length stand beside cells that a mirror replaces
    __device__ __forceinline__ void quad(float (&v)[4], int y, int z, int i) const {
        if (FROM == FROM_GRID || FROM == FROM_SUM) ld4a(v, o + a.g.row(y, z) + i);
        if (FROM == FROM_ZERO) v[0] = v[1] = v[2] = v[3] = 0.0f;
        if (FROM == FROM_COARSE || FROM == FROM_SUM) {
            // element i + j of either colour lies in coarse column i + j
            const float2 e = *reinterpret_cast<const float2*>(even_x(a.cg, c, y >> 1, z >> 1) + (i >> 1));
            const float2 d = *reinterpret_cast<const float2*>(odd_x(a.cg, c, y >> 1, z >> 1) + (i >> 1));
            const float cv[4] = {e.x, d.x, e.y, d.y};
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = FROM == FROM_SUM ? v[j] + cv[j] : cv[j];
        }
    }
    __device__ __forceinline__ float one(int y, int z, int i) const {
        float v = 0.0f;
        if (FROM == FROM_GRID || FROM == FROM_SUM) v = o[a.g.row(y, z) + i];
        if (FROM == FROM_COARSE || FROM == FROM_SUM) {
            const int k = clampi(i, 0, a.g.xs - 1);
            const float cv = ((k & 1) ? odd_x(a.cg, c, y >> 1, z >> 1) : even_x(a.cg, c, y >> 1, z >> 1))[k >> 1];
            v = FROM == FROM_SUM ? v + cv : cv;
        }
        return v;
    }
};

// A thread marches zc planes of one quad.  256^3 (134 MB): 27 us (5.0 TB/s), where
// the whole-grid kernels took 57.
// ADD: the last half-sweep of a cycle on the finest grid: f += v, and v itself
// is not stored.
template <int BLACK, int FROM, bool ADD>
__global__ void __launch_bounds__(256) k_gs_half(HalfArgs a) {
    int i, y;
    const Grid g = a.g;
    if (!quad_of(g.xs, g.d.Y - 2, i, y)) return;
    y += 1;
    const int X = g.d.X, Y = g.d.Y, Z = g.d.Z;
    const i64 sz = (i64)g.xs * Y;
    float* const v = a.v.p[blockIdx.z];
    const Other<FROM> o{v + (BLACK ? 0 : g.m), a.c.p[blockIdx.z], a};
    float* __restrict__ w = v + (BLACK ? g.m : 0);
    const float* __restrict__ rr = a.r.p[blockIdx.z] + (BLACK ? g.m : 0);
    const float* __restrict__ ss = a.s + (BLACK ? g.m : 0);
    const int z0 = 1 + blockIdx.y * a.zc, z1 = min(Z - 1, z0 + a.zc);
    float om[4], oc[4], op[4];
    i64 q = g.row(y, z0) + i;
    o.quad(om, y, z0 - 1, i);
    o.quad(oc, y, z0, i);
    for (int z = z0; z < z1; z++, q += sz) {
        const int e = ((y + z) & 1) ^ BLACK;  // the cells have x = 2 i + e
        float yp[4], ym[4], r4[4], s4[4], val[4];
        const float sc = o.one(y, z, e ? i + 4 : i - 1);
        o.quad(op, y, z + 1, i);
        o.quad(yp, y + 1, z, i);
        o.quad(ym, y - 1, z, i);
        ld4a(r4, rr + q);
        ld4a(s4, ss + q);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float side = e ? (j < 3 ? oc[j + 1] : sc) : (j > 0 ? oc[j - 1] : sc);
            float nb = oc[j] + side;
            nb = nb + yp[j];
            nb = nb + ym[j];
            nb = nb + op[j];
            nb = nb + om[j];
            val[j] = gs_value(nb, r4[j], s4[j], a.mu, a.h);
        }
        if (i == 0 && e == 0) val[0] = val[1];  // x = 0
        const int last = X - 1 - 2 * i - e;     // x = X - 1 is element last / 2
        if (last == 0) {                        // its mirror is in the quad before
            float nb = o.one(y, z, i - 1) + o.one(y, z, e ? i : i - 2);
            nb = nb + o.one(y + 1, z, i - 1);
            nb = nb + o.one(y - 1, z, i - 1);
            nb = nb + o.one(y, z + 1, i - 1);
            nb = nb + o.one(y, z - 1, i - 1);
            val[0] = gs_value(nb, rr[q - 1], ss[q - 1], a.mu, a.h);
        }
#pragma unroll
        for (int j = 1; j < 4; j++)
            if (last == 2 * j) val[j] = val[j - 1];
        // this cell's row and plane, and the boundary rows and planes it mirrors
        auto put = [&](int py, int pz) {
            if (!ADD) {
                st4a(w + g.row(py, pz) + i, val);
                return;
            }
            float* p = a.f.p[blockIdx.z] + g.d.at(2 * i, py, pz);
            float t[8];
            const bool whole = 2 * i + 7 < X;
            if (whole) __builtin_memcpy(t, p, 32);
            else
                for (int j = 0; j < 8; j++) t[j] = 2 * i + j < X ? p[j] : 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) t[j] = t[j] + (((j ^ e) & 1) ? oc[j >> 1] : val[j >> 1]);
            if (whole) __builtin_memcpy(p, t, 32);
            else
                for (int j = 0; j < 8; j++)
                    if (2 * i + j < X) p[j] = t[j];
        };
        auto rows_of = [&](int pz) {
            put(y, pz);
            if (y == 2) put(0, pz);
            if (y == Y - 3) put(Y - 1, pz);
        };
        rows_of(z);
        if (z == 2) rows_of(0);
        if (z == Z - 3) rows_of(Z - 1);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            om[j] = oc[j];
            oc[j] = op[j];
        }
    }
}

// restrictVolume, kernels_no_3d_write.cl:2218-2246: 2x2x2 mean, zero outside.
// A thread makes four coarse cells of a row; `row8(y, z, i, ev, od)` gives the
// eight fine values x = 2i .. 2i + 7 of a row.
template <class R>
__device__ __forceinline__ void restrict_quad(const Grid& f, const Grid& c, int i, int y, int z, float* out, R row8) {
    float ev[2][2][4], od[2][2][4];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const int Y = 2 * y + a, Z = 2 * z + b;
            if (2 * i < f.d.X && Y < f.d.Y && Z < f.d.Z) {
                row8(Y, Z, i, ev[a][b], od[a][b]);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (2 * (i + j) >= f.d.X) ev[a][b][j] = 0.0f;
                    if (2 * (i + j) + 1 >= f.d.X) od[a][b][j] = 0.0f;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) ev[a][b][j] = od[a][b][j] = 0.0f;
            }
        }
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float s = ev[0][0][j];
        s = s + od[0][0][j];
        s = s + ev[1][0][j];
        s = s + ev[0][1][j];
        s = s + od[1][0][j];
        s = s + ev[1][1][j];
        s = s + od[1][1][j];
        s = s + od[0][1][j];
        v[j] = 0.125f * s;
    }
    const int odd = (y + z) & 1;
    float* o = out + c.row(y, z) + (i >> 1);
    *reinterpret_cast<float2*>(o + (odd ? c.m : 0)) = make_float2(v[0], v[2]);
    *reinterpret_cast<float2*>(o + (odd ? 0 : c.m)) = make_float2(v[1], v[3]);
}

__global__ void __launch_bounds__(256) k_restrict(Trio fine, Grid f, Grid c, Trio coarse) {
    int i, y;
    if (!quad_of(c.d.X, c.d.Y, i, y)) return;
    const float* a = fine.p[blockIdx.z];
    restrict_quad(f, c, i, y, blockIdx.y, coarse.p[blockIdx.z], [&](int Y, int Z, int k, float* ev, float* od) {
        float t[4];
        ld4a(t, even_x(f, a, Y, Z) + k);
        __builtin_memcpy(ev, t, 16);
        ld4a(t, odd_x(f, a, Y, Z) + k);
        __builtin_memcpy(od, t, 16);
    });
}

// k_fmg_residual, restricted on the way.
__global__ void __launch_bounds__(256) k_fmg_residual_restrict(const float* __restrict__ Fc,
                                                               const float* __restrict__ f,
                                                               const float* __restrict__ s, Grid g, float mu,
                                                               float* __restrict__ r, Grid cg,
                                                               float* __restrict__ coarse) {
    int i, y;
    if (!quad_of(cg.d.X, cg.d.Y, i, y)) return;
    restrict_quad(g, cg, i, y, blockIdx.y, coarse, [&](int Y, int Z, int k, float* ev, float* od) {
        fmg_residual_row(Fc, f, s, g, mu, Y, Z, k, r, ev, od);
    });
}

// residual, kernels_no_3d_write.cl:2268-2301, restricted on the way.  (h h is
// a power of four: the product with its reciprocal rounds as the quotient.)
__device__ __forceinline__ float residual_of(float r, float s, float c, float nb, float mu, float ih2) {
    const float lap = (mu * (nb - 6.0f * c)) * ih2;
    return r - (lap - s * c);
}
__global__ void __launch_bounds__(256) k_residual_restrict(Trio v3, Trio r3, const float* __restrict__ s, Grid g,
                                                           Grid cg, float mu, float ih2, Trio coarse) {
    int i0, y0;
    if (!quad_of(cg.d.X, cg.d.Y, i0, y0)) return;
    const float *v = v3.p[blockIdx.z], *r = r3.p[blockIdx.z];
    const int X = g.d.X;
    restrict_quad(g, cg, i0, y0, blockIdx.y, coarse.p[blockIdx.z], [&](int Y, int Z, int i, float* ev, float* od) {
        const int y = remap(Y, g.d.Y), z = remap(Z, g.d.Z);
        const float *E = even_x(g, v, y, z) + i, *O = odd_x(g, v, y, z) + i;
        float e[4], o[4], a[4], b[4], c[4], d[4], re[4], se[4];
        ld4a(e, E);
        ld4a(o, O);
        ld4a(a, even_x(g, v, y + 1, z) + i);
        ld4a(b, even_x(g, v, y - 1, z) + i);
        ld4a(c, even_x(g, v, y, z + 1) + i);
        ld4a(d, even_x(g, v, y, z - 1) + i);
        ld4a(re, even_x(g, r, y, z) + i);
        ld4a(se, even_x(g, s, y, z) + i);
        const float before = O[-1], after = E[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float nb = o[j];
            nb = nb + (j ? o[j - 1] : before);
            nb = nb + a[j];
            nb = nb + b[j];
            nb = nb + c[j];
            nb = nb + d[j];
            ev[j] = residual_of(re[j], se[j], e[j], nb, mu, ih2);
        }
        ld4a(a, odd_x(g, v, y + 1, z) + i);
        ld4a(b, odd_x(g, v, y - 1, z) + i);
        ld4a(c, odd_x(g, v, y, z + 1) + i);
        ld4a(d, odd_x(g, v, y, z - 1) + i);
        ld4a(re, odd_x(g, r, y, z) + i);
        ld4a(se, odd_x(g, s, y, z) + i);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float nb = j < 3 ? e[j + 1] : after;
            nb = nb + e[j];
            nb = nb + a[j];
            nb = nb + b[j];
            nb = nb + c[j];
            nb = nb + d[j];
            od[j] = residual_of(re[j], se[j], o[j], nb, mu, ih2);
        }
        if (i == 0) ev[0] = ev[1];     // x = 0
        const int last = X - 1 - 2 * i;  // x = X - 1
        if (last == 0 || last == 1) {  // its mirror X - 3 is in the quad before
            const bool odd = last == 1;
            const float *C = (odd ? O : E) - 1, *N = odd ? E : O;  // N: the row's other colour
            const float* a4[4] = {odd ? odd_x(g, v, y + 1, z) : even_x(g, v, y + 1, z),
                                  odd ? odd_x(g, v, y - 1, z) : even_x(g, v, y - 1, z),
                                  odd ? odd_x(g, v, y, z + 1) : even_x(g, v, y, z + 1),
                                  odd ? odd_x(g, v, y, z - 1) : even_x(g, v, y, z - 1)};
            float nb = odd ? N[0] : N[-1];
            nb = nb + (odd ? N[-1] : N[-2]);
            for (int k = 0; k < 4; k++) nb = nb + a4[k][i - 1];
            const float rv = (odd ? odd_x(g, r, y, z) : even_x(g, r, y, z))[i - 1];
            const float sv = (odd ? odd_x(g, s, y, z) : even_x(g, s, y, z))[i - 1];
            (odd ? od : ev)[0] = residual_of(rv, sv, C[0], nb, mu, ih2);
        }
#pragma unroll
        for (int j = 1; j < 4; j++) {
            if (last == 2 * j) ev[j] = ev[j - 1];
            if (last == 2 * j + 1) od[j] = od[j - 1];
        }
    });
}

// prolongate (ADD) / prolongate2 where no sweep follows.
template <bool ADD>
__global__ void __launch_bounds__(256) k_prolong(Trio coarse, Grid c, Grid f, Trio fine) {
    int i, y;
    if (!quad_of(f.xs, f.d.Y, i, y)) return;
    const int z = blockIdx.y;
    const float2 e = *reinterpret_cast<const float2*>(even_x(c, coarse.p[blockIdx.z], y >> 1, z >> 1) + (i >> 1));
    const float2 o = *reinterpret_cast<const float2*>(odd_x(c, coarse.p[blockIdx.z], y >> 1, z >> 1) + (i >> 1));
    const float cv[4] = {e.x, o.x, e.y, o.y};
#pragma unroll
    for (int b = 0; b < 2; b++) {
        float* p = fine.p[blockIdx.z] + f.row(y, z) + i + (b ? f.m : 0);
        float v[4];
        if (ADD) ld4a(v, p);
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = ADD ? v[j] + cv[j] : cv[j];
        st4a(p, v);
    }
}

// f += e on the finest grid where no sweep ends a cycle; f is a plain array
__global__ void __launch_bounds__(256) k_add_inplace(float* __restrict__ f, const float* __restrict__ e, Grid g) {
    int i, y;
    if (!quad_of(g.xs, g.d.Y, i, y)) return;
    const int z = blockIdx.y;
    float ev[4], od[4];
    ld4a(ev, even_x(g, e, y, z) + i);
    ld4a(od, odd_x(g, e, y, z) + i);
    float* p = f + g.d.at(2 * i, y, z);
    if (2 * i + 7 < g.d.X) {
        float t[8];
        __builtin_memcpy(t, p, 32);
#pragma unroll
        for (int j = 0; j < 8; j++) t[j] = t[j] + ((j & 1) ? od[j >> 1] : ev[j >> 1]);
        __builtin_memcpy(p, t, 32);
    } else {
        for (int j = 0; j < 8; j++)
            if (2 * i + j < g.d.X) p[j] = p[j] + ((j & 1) ? od[j >> 1] : ev[j >> 1]);
    }
}

// n quads of each array
__global__ void __launch_bounds__(256) k_zero(Trio v, i64 n) {
    float4* p = reinterpret_cast<float4*>(v.p[blockIdx.z]);
    for (i64 i = blockIdx.x * (i64)256 + threadIdx.x; i < n; i += (i64)gridDim.x * 256) p[i] = make_float4(0, 0, 0, 0);
}
__global__ void k_fill(float* __restrict__ p, i64 n, float v) {
    for (i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x) p[i] = v;
}

// MGGVFFinish, kernels_no_3d_write.cl:2202-2216: w = |v|, no zero guard.
__global__ void k_fmg_finish(const float* __restrict__ x, const float* __restrict__ y, const float* __restrict__ z,
                             float* __restrict__ w, i64 n) {
    for (i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x)
        w[i] = sqrtf(x[i] * x[i] + y[i] * y[i] + z[i] * z[i]);
}

// Sum of squares in double: per-block partials, then one block folds them.
__global__ void __launch_bounds__(256) k_sumsq_partial(const float* __restrict__ a, i64 n, double* __restrict__ part) {
    __shared__ double sh[256];
    double s = 0.0;
    for (i64 i = blockIdx.x * (i64)blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x) {
        double v = (double)a[i];
        s += v * v;
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}
__global__ void __launch_bounds__(256) k_sum_partials(const double* __restrict__ part, int n, double* __restrict__ out) {
    __shared__ double sh[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += part[i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = sh[0];
}
constexpr int NPART = 1024;

static unsigned g1(i64 n) {
    i64 g = (n + 255) / 256;
    return (unsigned)(g > 16384 ? 16384 : (g < 1 ? 1 : g));
}

static Dims coarser(Dims d) {
    int m = d.X > d.Y ? d.X : d.Y;
    m = m > d.Z ? m : d.Z;
    int p = 1;
    while (p < m) p *= 2;
    int s = p / 2 > 1 ? p / 2 : 1;
    return Dims{s, s, s};
}

struct Level {
    Grid g;
    Trio r, v;
    float* s;
};

// cells up to which a level runs its components in one launch
constexpr i64 FMG_WIDE = (i64)1 << 22;
// cells of the finest grid up to which all three components have buffers
constexpr i64 FMG_TOGETHER = (i64)1 << 27;

struct Solver {
    std::vector<Level> L;
    float mu;
    int v0, v1, v2;
    int comps;  // components per cycle
    Trio f;     // and their f
    hipStream_t st;
    tsf_status err = TSF_OK;

    void chk() {
        if (err == TSF_OK) err = check_launch("tsf_gvf_fmg");
    }
    static Trio from(const Trio& t, int c) { return Trio{{t.p[c], t.p[c < 2 ? c + 1 : 2], t.p[2]}}; }
    // f(c, n): n components from c, all in one launch or one by one
    template <class F>
    void split(int l, F f) {
        if (L[l].g.d.n() <= FMG_WIDE) f(0, comps);
        else
            for (int c = 0; c < comps; c++) f(c, 1);
    }
    // v as `from` says, where no sweep follows
    void set(int l, int c, int n, int from) {
        Level& a = L[l];
        if (from == FROM_ZERO) {
            const i64 quads = 2 * a.g.m / 4;
            hipLaunchKernelGGL(k_zero, dim3(g1(quads), 1, n), 256, 0, st, Solver::from(a.v, c), quads);
        } else if (from != FROM_GRID) {
            Level& b = L[l + 1];
            const dim3 gr = quad_grid(a.g.xs, a.g.d.Y, a.g.d.Z, n);
            const Trio cv = Solver::from(b.v, c), fv = Solver::from(a.v, c);
            if (from == FROM_SUM) hipLaunchKernelGGL(k_prolong<true>, gr, 256, 0, st, cv, b.g, a.g, fv);
            else hipLaunchKernelGGL(k_prolong<false>, gr, 256, 0, st, cv, b.g, a.g, fv);
        }
        chk();
    }
    // sweeps on v, which starts as `from` says; add: the last one ends in f += v
    void smooth(int l, int c, int n, int iters, int from, bool add) {
        if (iters == 0) {
            set(l, c, n, from);
            if (add)
                for (int k = c; k < c + n; k++)
                    hipLaunchKernelGGL(k_add_inplace, quad_grid(L[0].g.xs, L[0].g.d.Y, L[0].g.d.Z, 1), 256, 0, st, f.p[k],
                                       L[0].v.p[k], L[0].g);
            chk();
            return;
        }
        Level &a = L[l], &b = L[l + 1 < (int)L.size() ? l + 1 : l];
        const int planes = a.g.d.Z - 2;
        // planes per thread: the neighbour planes stay in registers, but 2048
        // workgroups (8 per compute unit) come first
        int zc = 8;
        while (zc > 1 && (i64)quad_grid(a.g.xs, a.g.d.Y - 2, 1, n).x * n * ((planes + zc - 1) / zc) < 2048) zc /= 2;
        const dim3 gr = quad_grid(a.g.xs, a.g.d.Y - 2, (planes + zc - 1) / zc, n);
        const HalfArgs h{Solver::from(a.v, c), Solver::from(a.r, c), a.s, a.g, mu, (float)(1 << l), zc,
                         Solver::from(b.v, c), b.g, Solver::from(f, c)};
        for (int i = 0; i < iters; i++) {
            switch (i == 0 ? from : FROM_GRID) {
                case FROM_GRID: hipLaunchKernelGGL((k_gs_half<0, FROM_GRID, false>), gr, 256, 0, st, h); break;
                case FROM_COARSE: hipLaunchKernelGGL((k_gs_half<0, FROM_COARSE, false>), gr, 256, 0, st, h); break;
                case FROM_SUM: hipLaunchKernelGGL((k_gs_half<0, FROM_SUM, false>), gr, 256, 0, st, h); break;
                default: hipLaunchKernelGGL((k_gs_half<0, FROM_ZERO, false>), gr, 256, 0, st, h);
            }
            if (add && i + 1 == iters) hipLaunchKernelGGL((k_gs_half<1, FROM_GRID, true>), gr, 256, 0, st, h);
            else hipLaunchKernelGGL((k_gs_half<1, FROM_GRID, false>), gr, 256, 0, st, h);
            chk();
        }
    }
    void vcycle(int l, int from, bool add) {
        const bool last = l + 1 == (int)L.size();
        split(l, [&](int c, int n) {
            Level& a = L[l];
            smooth(l, c, n, v1, from, false);
            if (last) {
                smooth(l, c, n, v2, FROM_GRID, add);
                return;
            }
            Level& b = L[l + 1];
            const float h = (float)(1 << l);
            hipLaunchKernelGGL(k_residual_restrict, quad_grid(b.g.d.X, b.g.d.Y, b.g.d.Z, n), 256, 0, st,
                               Solver::from(a.v, c), Solver::from(a.r, c), a.s, a.g, b.g, mu, 1.0f / (h * h),
                               Solver::from(b.r, c));
            chk();
        });
        if (last) return;
        vcycle(l + 1, FROM_ZERO, false);
        split(l, [&](int c, int n) { smooth(l, c, n, v2, FROM_SUM, add); });
    }
    // level l from its r; on level 0, whose r is restricted already, f += v
    void fmg(int l) {
        int from = FROM_ZERO;
        if (l + 1 < (int)L.size()) {
            if (l > 0)
                split(l, [&](int c, int n) {
                    Level &a = L[l], &b = L[l + 1];
                    hipLaunchKernelGGL(k_restrict, quad_grid(b.g.d.X, b.g.d.Y, b.g.d.Z, n), 256, 0, st,
                                       Solver::from(a.r, c), a.g, b.g, Solver::from(b.r, c));
                    chk();
                });
            fmg(l + 1);
            from = FROM_COARSE;
        }
        for (int i = 0; i < v0; i++) vcycle(l, i == 0 ? from : FROM_GRID, l == 0 && i + 1 == v0);
        if (v0 == 0) split(l, [&](int c, int n) { smooth(l, c, n, 0, from, l == 0); });
    }
};

static std::vector<Dims> level_dims(Dims d, int levels) {
    std::vector<Dims> v{d};
    for (int l = 0; l < levels; l++) v.push_back(coarser(v.back()));
    return v;
}

// a colour-split array of one grid
static size_t array_bytes(const Grid& g) { return ((size_t)g.m * 8 + 255) & ~(size_t)255; }
// the workspace: r and v per component and s, of every level
static size_t fmg_bytes(const std::vector<Dims>& levels, int comps) {
    size_t b = 0;
    for (Dims d : levels) b += (2 * comps + 1) * array_bytes(Grid(d));
    return b + NPART * sizeof(double) + 256;
}
// five plain arrays of every level: what callers were told while the grids
// were whole, more than one component needs but for rows of 4 or 9 elements
// (their padding) and a few smallest volumes (the arrays' alignment)
static size_t five_grids_bytes(const std::vector<Dims>& levels) {
    size_t b = 0;
    for (Dims d : levels) b += 5 * (((size_t)d.n() * 4 + 255) & ~(size_t)255);
    return b + NPART * sizeof(double) + 256;
}

}  // namespace tsf

using namespace tsf;

extern "C" {

size_t tsf_gvf_fmg_workspace_size(tsf_dims dims, int32_t levels) {
    if (levels < 0 || levels > 12) return 0;
    return fmg_bytes(level_dims(D(dims), levels), D(dims).n() <= FMG_TOGETHER ? 3 : 1);
}

tsf_status tsf_gvf_fmg(const tsf_field* f, const tsf_field* out, tsf_dims dims, float mu, int32_t iterations,
                       int32_t levels, int32_t v0, int32_t v1, int32_t v2, double* residual_norms, void* workspace,
                       size_t workspace_bytes, hipStream_t stream) {
    const char* W = "tsf_gvf_fmg";
    TSF_TRY(check_field(f, false, W));
    TSF_TRY(check_field(out, true, W));
    if (f->storage != TSF_STORAGE_F32 || out->storage != TSF_STORAGE_F32)
        return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: FMG supports F32 storage only", W);
    TSF_TRY(check_dims(dims, 4, W));
    if (iterations < 0 || levels < 0 || levels > 12 || v0 < 0 || v1 < 0 || v2 < 0)
        return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: negative iteration, level or sweep count", W);
    if (!(mu > 0.0f) || !__builtin_isfinite(mu)) return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: mu must be > 0", W);
    std::vector<Dims> ld = level_dims(D(dims), levels);
    if (ld.back().X < 4) return set_error(TSF_ERR_DIMENSIONS, "%s: coarsest grid below 4^3", W);
    if (f->x == out->x || f->y == out->y || f->z == out->z)
        return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: f and out planes must not alias", W);
    Scratch sc;
    // a workspace, or a device, short of three components' arrays runs them one
    // by one; a workspace of five plain arrays too small even for that is
    // accepted and not used
    const size_t one = fmg_bytes(ld, 1), three = fmg_bytes(ld, 3);
    bool together = D(dims).n() <= FMG_TOGETHER;
    if (workspace) {
        together = together && workspace_bytes >= three;
        TSF_TRY(sc.get(workspace, workspace_bytes, std::min(one, five_grids_bytes(ld)), W));
        if (workspace_bytes < one) TSF_TRY(sc.get(nullptr, 0, one, W));
    } else {
        together = together && sc.get(nullptr, 0, three, W) == TSF_OK;
        if (!together) TSF_TRY(sc.get(nullptr, 0, one, W));
    }
    Solver S;
    S.mu = mu;
    S.v0 = v0;
    S.v1 = v1;
    S.v2 = v2;
    S.comps = together ? 3 : 1;
    S.st = stream;
    char* p = (char*)sc.ptr;
    for (Dims d : ld) {
        Level lv{Grid(d), {}, {}, nullptr};
        const size_t b = array_bytes(lv.g);
        auto next = [&] {
            float* q = (float*)p;
            p += b;
            return q;
        };
        for (int c = 0; c < 3; c++) {
            lv.r.p[c] = c < S.comps ? next() : lv.r.p[0];
            lv.v.p[c] = c < S.comps ? next() : lv.v.p[0];
        }
        lv.s = next();
        S.L.push_back(lv);
    }
    double* part = (double*)p;
    double* norm_out = part + NPART;
    const float* F[3] = {(const float*)f->x, (const float*)f->y, (const float*)f->z};
    float* O[3] = {(float*)out->x, (float*)out->y, (float*)out->z};
    const Grid g0 = S.L[0].g;
    const i64 n0 = g0.d.n();
    const dim3 gr0 = quad_grid(g0.xs, g0.d.Y, g0.d.Z, 1);
    // |F|^2 at every level (restricted once)
    hipLaunchKernelGGL(k_sqrmag, gr0, 256, 0, stream, F[0], F[1], F[2], g0, S.L[0].s);
    S.chk();
    for (size_t l = 1; l < S.L.size(); l++) {
        const Grid &a = S.L[l - 1].g, &b = S.L[l].g;
        hipLaunchKernelGGL(k_restrict, quad_grid(b.d.X, b.d.Y, b.d.Z, 1), 256, 0, stream,
                           Trio{{S.L[l - 1].s, nullptr, nullptr}}, a, b, Trio{{S.L[l].s, nullptr, nullptr}});
    }
    S.chk();
    for (int c0 = 0; c0 < 3 && S.err == TSF_OK; c0 += S.comps) {
        for (int k = 0; k < S.comps; k++)
            hipLaunchKernelGGL(k_fill, g1(n0), 256, 0, stream, O[c0 + k], n0, 0.0f);
        S.chk();
        for (int it = 0; it < iterations && S.err == TSF_OK; it++) {
            for (int k = 0; k < S.comps; k++) {
                const int c = c0 + k;
                S.f.p[k] = O[c];
                if (S.L.size() > 1) {
                    const Level& b = S.L[1];
                    hipLaunchKernelGGL(k_fmg_residual_restrict, quad_grid(b.g.d.X, b.g.d.Y, b.g.d.Z, 1), 256, 0, stream,
                                       F[c], O[c], S.L[0].s, g0, mu, S.L[0].r.p[k], b.g, b.r.p[k]);
                } else {
                    hipLaunchKernelGGL(k_fmg_residual, gr0, 256, 0, stream, F[c], O[c], S.L[0].s, g0, mu,
                                       S.L[0].r.p[k]);
                }
                S.chk();
                if (residual_norms) {
                    hipLaunchKernelGGL(k_sumsq_partial, NPART, 256, 0, stream, S.L[0].r.p[k], 2 * g0.m, part);
                    hipLaunchKernelGGL(k_sum_partials, 1, 256, 0, stream, part, NPART, norm_out);
                    S.chk();
                    double ss = 0.0;
                    hipError_t e = hipMemcpyAsync(&ss, norm_out, sizeof ss, hipMemcpyDeviceToHost, stream);
                    if (e == hipSuccess) e = hipStreamSynchronize(stream);
                    if (e != hipSuccess) return set_error(TSF_ERR_HIP, "%s: %s", W, hipGetErrorString(e));
                    residual_norms[c * iterations + it] = sqrt(ss);
                }
            }
            S.fmg(0);
        }
    }
    if (S.err != TSF_OK) return S.err;
    hipLaunchKernelGGL(k_fmg_finish, g1(n0), 256, 0, stream, O[0], O[1], O[2], (float*)out->w, n0);
    TSF_TRY(check_launch(W));
    if (sc.owned) {
        hipError_t e = hipStreamSynchronize(stream);
        if (e != hipSuccess) return set_error(TSF_ERR_HIP, "%s: %s", W, hipGetErrorString(e));
    }
    return TSF_OK;
}

}  // extern "C"
