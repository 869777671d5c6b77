// K reverse steps of the gradient vector flow per launch: the transpose of
// k_gvf_cols's march (gvf_cols.hpp).
//
//   in   L = fold(lam^{n+1}), zero on every boundary plane; v[k] = v^{n-k},
//        k = 0 .. K-1; F; dF
//   out  fold(lam^{n-K+1}), or with !FOLD (the launch ends at v^0 = f)
//        dF += lam^0
//   dF  += the data-term gradients of the K steps
//   part[b] += block b's share of d/dmu of the K steps
//
// One step: lam = (1 - 6 mu - |f|^2) L + mu nb(L), nb the sum over the six
// neighbours, and its fold, lam + mu e at interior voxels and 0 elsewhere,
// where e adds the neighbour on the boundary side for a voxel two planes from
// a face (the boundary voxel it mirrors into has no other contribution).  The
// data term gives dF += L |f|^2 + 2 f sum_c L_c (f_c - v_c), and d/dmu is the
// sum over every voxel of v . (nb - 6 L) (k_gvf_adj_march says why), here as
// fused multiply-adds in double of two floats: their products are exact, so
// they round as products and sums do.  Expressions and their order are those
// of k_gvf_adj_march: one launch and K of that one give the same adjoint and
// dF bit for bit.
//
// A workgroup of NW waves covers 64 x NW columns, a wave per row.  Stage k
// turns plane t - k of L into that plane of the next adjoint; x neighbours
// come by DPP shifts, y neighbours through LDS (each wave publishes its row
// of each new plane, one barrier per step), z neighbours from registers.  The
// adjoint is zero outside the interior, so tiles need no halo at the volume's
// sides; elsewhere stage k is valid on the tile less k + 1 columns and k rows
// at each side.  Every voxel is owned by one tile: where the last tile is
// shifted to end at the volume's edge, the columns and rows of the one before
// are not its own.  States and dF are read on owned voxels only; elsewhere
// their loads are past the resource, which costs no memory access, and read 0.
//
// What bounds it: HBM, 60 + 12 K bytes a voxel for K steps, and on small
// volumes a step's latency.  Per reverse step, against the earlier two-step
// kernel on 64-plane chunks and the reductions after each of its launches:
// 64^3 56 -> 6.8 us, 128^3 58 -> 21, 256^3 244 -> 153, 512^3 1581 -> 1118
// (3.84 TB/s).  The branch on the fold is taken per step, not per stage: in
// the stages it cost 70 registers.
#pragma once

#include "gvf_cols.hpp"

namespace tsf {

template <int K>
struct AdjColsArgs {
    const float* L;
    const float* v[K];
    const float* f[3];
    float* out;
    float* dF;
    double* part;
    Dims d;
    float mu;
    int zc;
};

template <int K, int NW, bool FOLD>
struct AdjCols {
    static constexpr int OW = 64 - 2 * K, OH = NW - 2 * (K - 1);
    struct Lds {
        // the waves' rows of each adjoint, the rows above and below the tile
        // (zero but for L's), and one that is not read
        float row[K][3][NW + 3][64];
    };

    const AdjColsArgs<K>& a;
    Lds* S;
    int lane, w, cy, q0, q1, xfold, yfold;
    bool inter, fx2, fxN;
    unsigned cb, pb, col, hcol, ocol;  // bytes per volume and plane; cell offsets (ocol: NO_LANE where not owned)
    int pub, pdn, pup, pring;  // LDS words of this wave's row, its neighbours' and its ring row
    __amdgpu_buffer_rsrc_t rL, rd, ro, rf[3], rv[K];

    float l0[4][3], hr[2][3], fr[4][3], vr[K][3], dr[3];
    float P[K][3], C[K][3], fd[K][3], g[K][3];
    double gm;

    __device__ __forceinline__ AdjCols(const AdjColsArgs<K>& args, Lds* lds) : a(args), S(lds) {}

    static __device__ __forceinline__ float ld(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)v, (int)s, 0));
    }
    // plane z of a volume: its offset, and the mask that drops the access when
    // z is outside [lo, hi)
    __device__ __forceinline__ unsigned zoff(int z) const { return (unsigned)clampi(z, 0, a.d.Z - 1) * pb; }
    static __device__ __forceinline__ unsigned drop(int z, int lo, int hi) { return z >= lo && z < hi ? 0u : NO_LANE; }

    __device__ __forceinline__ void load_l(float (&q)[3], unsigned at, int z) {
        const unsigned s = zoff(z), v = at | drop(z, 0, a.d.Z);
#pragma unroll
        for (int c = 0; c < 3; c++) q[c] = ld(rL, v, c * cb + s);
    }
    __device__ __forceinline__ void load_f(float (&q)[3], int z) {
        const unsigned s = zoff(z);
#pragma unroll
        for (int c = 0; c < 3; c++) q[c] = ld(rf[c], col, s);
    }
    __device__ __forceinline__ void load_own(__amdgpu_buffer_rsrc_t r, float (&q)[3], int z) {
        const unsigned s = zoff(z), v = ocol | drop(z, q0, q1);
#pragma unroll
        for (int c = 0; c < 3; c++) q[c] = ld(r, v, c * cb + s);
    }

    template <int U, bool EDGE>
    __device__ __forceinline__ void step(int t) {
        constexpr int bw = U & 1, br = bw ^ 1;
        const int Z = a.d.Z;
        float N[3];
#pragma unroll
        for (int k = K - 1; k >= 1; k--)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                fd[k][c] = fd[k - 1][c];
                g[k][c] = g[k - 1][c];
            }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            N[c] = l0[(U + 1) & 3][c];
            fd[0][c] = fr[U & 3][c];
            g[0][c] = dr[c];
            S[bw].row[0][c][0][pub] = N[c];
            S[bw].row[0][c][0][pring] = hr[U & 1][c];
        }
        load_own(rd, dr, t + 1);
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int p = t - k;
            float yp[3], ym[3], nb[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                ym[c] = S[br].row[k][c][0][pdn];
                yp[c] = S[br].row[k][c][0][pup];
            }
#pragma unroll
            for (int c = 0; c < 3; c++) nb[c] = lane_right(C[k][c]);
            __builtin_amdgcn_sched_barrier(NOT_VALU);
#pragma unroll
            for (int c = 0; c < 3; c++) nb[c] = nb[c] + lane_left(C[k][c]);
            __builtin_amdgcn_sched_barrier(NOT_VALU);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                nb[c] = nb[c] + yp[c];
                nb[c] = nb[c] + ym[c];
                nb[c] = nb[c] + N[c];
                nb[c] = nb[c] + P[k][c];
            }
            const float* f = fd[k];
            const float m2 = f[0] * f[0] + f[1] * f[1] + f[2] * f[2];
            const float diag = 1.0f - 6.0f * a.mu - m2;
            float lam[3], o[3], s = 0.0f;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                lam[c] = diag * C[k][c] + a.mu * nb[c];
                s += C[k][c] * (f[c] - vr[k][c]);
                gm = __builtin_fma((double)vr[k][c], (double)(nb[c] - 6.0f * C[k][c]), gm);
                o[c] = lam[c];
            }
            if (EDGE) {
                const bool fy2 = cy == 2, fyN = cy == a.d.Y - 3, fz2 = p == 2, fzN = p == Z - 3;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const float lxm = lane_left(C[k][c]), lxp = lane_right(C[k][c]);
                    const float e = (fx2 ? lxm : 0.0f) + (fxN ? lxp : 0.0f) + (fy2 ? ym[c] : 0.0f) +
                                    (fyN ? yp[c] : 0.0f) + (fz2 ? P[k][c] : 0.0f) + (fzN ? N[c] : 0.0f);
                    o[c] = lam[c] + a.mu * e;
                }
            }
            const bool in = inter && p >= 1 && p <= Z - 2;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                o[c] = in ? o[c] : 0.0f;
                g[k][c] = g[k][c] + (C[k][c] * m2 + 2.0f * f[c] * s);
                if (k < K - 1) S[bw].row[k + 1][c][0][pub] = o[c];
            }
            if (k == K - 1) {
                const unsigned so = zoff(p), vo = ocol | drop(p, q0, q1);
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const float q = FOLD ? g[k][c] : g[k][c] + lam[c];
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(q), rd, (int)vo, (int)(c * cb + so), 0);
                    if (FOLD)
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[c]), ro, (int)vo, (int)(c * cb + so), 0);
                }
            }
            load_own(rv[k], vr[k], p + 1);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                P[k][c] = C[k][c];
                C[k][c] = N[c];
                N[c] = o[c];
            }
            if (k == 0) {
                load_l(l0[(U + 3) & 3], col, t + 3);
                load_l(hr[U & 1], hcol, t + 3);
            }
        }
        load_f(fr[(U + 2) & 3], t + 2);
        __syncthreads();
    }

    // whether a stage of step t folds: the tile or the wave's row lies two from
    // a face, or a stage's plane does
    __device__ __forceinline__ bool edge(int t) const {
        return xfold + yfold != 0 || (t >= 2 && t <= K + 1) || (t >= a.d.Z - 3 && t <= a.d.Z + K - 4);
    }

    __device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(const void* p, unsigned bytes) const {
        int n = __builtin_amdgcn_readfirstlane((int)bytes), f = BUFFER_WORD3;
        asm volatile("" : "+s"(n), "+s"(f));
        return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, n, f);
    }

    __device__ __forceinline__ void run() {
        const Dims d = a.d;
        lane = threadIdx.x & 63;
        w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        int tbx, tby, tbz;
        xcd_tile(tbx, tby, tbz);
        tbx = __builtin_amdgcn_readfirstlane(tbx);
        tby = __builtin_amdgcn_readfirstlane(tby);
        tbz = __builtin_amdgcn_readfirstlane(tbz);
        const int ex = max(min(tbx * OW, d.X - 64), 0), ey = max(min(tby * OH, d.Y - NW), 0);
        const int cx = ex + lane;
        cy = ey + w;
        q0 = tbz * a.zc;
        q1 = min(q0 + a.zc, d.Z);
        pb = (unsigned)d.X * (unsigned)d.Y * 4u;
        cb = pb * (unsigned)d.Z;
        const bool act = cx < d.X && cy < d.Y;
        const unsigned at = (unsigned)(cy * d.X + cx) * 4u;
        col = act ? at : NO_LANE;
        const bool own = act && (tbx == 0 || cx >= tbx * OW + K) && (lane < 64 - K || ex + 64 >= d.X) &&
                         (tby == 0 || cy >= tby * OH + K - 1) && (w < NW - (K - 1) || ey + NW >= d.Y);
        ocol = own ? at : NO_LANE;
        hcol = NO_LANE;
        if (w == 0 && ey > 0 && cx < d.X) hcol = (unsigned)((ey - 1) * d.X + cx) * 4u;
        if (w == NW - 1 && ey + NW < d.Y && cx < d.X) hcol = (unsigned)((ey + NW) * d.X + cx) * 4u;
        inter = cx >= 1 && cx <= d.X - 2 && cy >= 1 && cy <= d.Y - 2;
        fx2 = cx == 2;
        fxN = cx == d.X - 3;
        xfold = __builtin_amdgcn_readfirstlane(ex <= 2 || ex + 63 >= d.X - 3);
        yfold = __builtin_amdgcn_readfirstlane(cy == 2 || cy == d.Y - 3);
        pub = w * 64 + lane;
        pdn = (w == 0 ? NW : w - 1) * 64 + lane;
        pup = (w == NW - 1 ? NW + 1 : w + 1) * 64 + lane;
        pring = (w == 0 ? NW : (w == NW - 1 ? NW + 1 : NW + 2)) * 64 + lane;
        rL = resource(a.L, 3u * cb);
        rd = resource(a.dF, 3u * cb);
        ro = resource(FOLD ? a.out : a.dF, 3u * cb);
#pragma unroll
        for (int c = 0; c < 3; c++) rf[c] = resource(a.f[c], cb);
#pragma unroll
        for (int k = 0; k < K; k++) rv[k] = resource(a.v[k], 3u * cb);
        gm = 0.0;
        const int t0 = q0 - (K - 1), te = q1 + K - 2;
        float qh[3];
#pragma unroll
        for (int i = 0; i < 4; i++) load_l(l0[(i + 3) & 3], col, t0 - 1 + i);
        load_l(qh, hcol, t0);
        load_l(hr[0], hcol, t0 + 1);
        load_l(hr[1], hcol, t0 + 2);
        load_f(fr[0], t0);
        load_f(fr[1], t0 + 1);
        load_own(rd, dr, t0);
#pragma unroll
        for (int k = 0; k < K; k++) {
            load_own(rv[k], vr[k], t0 - k);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                P[k][c] = k == 0 ? l0[3][c] : 0.0f;
                C[k][c] = k == 0 ? l0[0][c] : 0.0f;
                fd[k][c] = g[k][c] = 0.0f;
            }
        }
        for (int i = threadIdx.x; i < (int)(2 * sizeof(Lds) / 4); i += 64 * NW) (&S[0].row[0][0][0][0])[i] = 0.0f;
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 3; c++) {
            S[1].row[0][c][0][pub] = C[0][c];
            S[1].row[0][c][0][pring] = qh[c];
        }
        __syncthreads();
        for (int t = t0; t <= te; t += 4) {
            if (edge(t)) step<0, true>(t);
            else step<0, false>(t);
            if (edge(t + 1)) step<1, true>(t + 1);
            else step<1, false>(t + 1);
            if (edge(t + 2)) step<2, true>(t + 2);
            else step<2, false>(t + 2);
            if (edge(t + 3)) step<3, true>(t + 3);
            else step<3, false>(t + 3);
        }
    }
};

template <int K, int NW, int WPE, bool FOLD>
__global__ void __launch_bounds__(64 * NW, WPE) k_gvf_adj_cols(AdjColsArgs<K> a) {
    typedef AdjCols<K, NW, FOLD> M;
    __shared__ typename M::Lds lds[2];
    __shared__ double red[NW];
    M m(a, lds);
    m.run();
    // the block's sum in a fixed order: within each wave by xor shuffles,
    // then the waves in order
    double s = m.gm;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double sum = 0.0;
#pragma unroll
        for (int i = 0; i < NW; i++) sum += red[i];
        a.part[blockIdx.x + (i64)gridDim.x * (blockIdx.y + (i64)gridDim.y * blockIdx.z)] += sum;
    }
}

}  // namespace tsf
