// K Jacobi steps of the gradient vector flow per launch.
//
// v and f cross HBM once per K iterations.  A workgroup of NW waves covers a
// tile of 64 x (NW * R) columns: lane l of wave w owns column ex + l of the R
// rows ey + w R ..., and the workgroup marches a chunk of zc planes.  Stage k
// (0 .. K-1) turns plane t - k of iterate k into that plane of iterate k + 1,
// so one plane of the result leaves the pipeline per step of t.  Of iterate k
// a thread keeps two planes (the one below and the one being updated); the
// third arrives from stage k - 1, or from memory for k = 0.
//   - x neighbours come across lanes by DPP wave shifts, which the adds take
//     as an operand;
//   - y neighbours inside a thread's R rows are registers; those of the first
//     and last row come through LDS, where every wave publishes these two rows
//     of each new plane (double buffered: one barrier per step);
//   - z neighbours are registers.
// Stage k is valid on the tile less k + 1 columns at each side and, since the
// rows just above and below the tile are loaded for stage 0, less k rows: the
// output tile is (64 - 2K) x (NW R - 2K + 2).  Invalid rows and lanes compute
// on whatever they hold and store nothing.
//
// Mirror rule (kernels_no_3d_write.cl:1757-1760): the value at w is the update
// at mirror(w), 0 -> 2 and N-1 -> N-3.  For the iterates after the first, the
// neighbour of voxel 1 on the boundary side therefore equals its neighbour on
// the other side (likewise N-2).  In z and y the sums read the other neighbour
// there (uniform branches), in x the boundary lanes take their mirror's value.
// The launch also stores the faces: x faces from their lanes, y and z faces by
// the thread that computes the mirror.
//
// What bounds it: at 256^3 and below the issue of a step's instructions and
// its latency (barrier, LDS, the chain through the stages: 0.8 us a step for
// 8 rows and two stages, where its arithmetic takes 0.3); above, that and HBM.
// Against the earlier two- and four-step kernels (x neighbours through LDS,
// 64-plane chunks at every size, a second launch for the faces), per
// iteration: F32 64^3 22.6 -> 4.4 us, 128^3 26.6 -> 11.1, 256^3 93 -> 56,
// 512^3 545 -> 401; SNORM16 301 x 247 x 329 113 -> 83, 512^3 504 -> 412.
// Loads further ahead and two or three rows per thread at K = 3 measured the
// same or slower.
//
// The arithmetic runs on stored numbers (value * unit, unit a power of two),
// so it rounds as on the values; operation order is the reference's, so K
// steps in one launch equal K launches bit for bit where the middle iterates
// are not rounded (F32) or are rounded alike (SNORM16).
#pragma once

#include <math.h>

#include "tsf_common.hpp"

namespace tsf {

// The stored number of one element: getu() reads it as a float in storage
// units, put() stores a float given in units, bload() and bstore() are raw
// buffer accesses.
template <class S>
struct Raw;
template <>
struct Raw<F32> {
    typedef float T;
    static __device__ __forceinline__ float getu(T r) { return r; }
    static __device__ __forceinline__ T put(float u) { return u; }
    static __device__ __forceinline__ T bload(__amdgpu_buffer_rsrc_t b, unsigned v, unsigned s) {
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, (int)v, (int)s, 0));
    }
    static __device__ __forceinline__ void bstore(__amdgpu_buffer_rsrc_t b, T q, unsigned v, unsigned s) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(q), b, (int)v, (int)s, 0);
    }
};
template <>
struct Raw<F16> {
    typedef unsigned short T;
    static __device__ __forceinline__ float getu(T r) { return __half2float(__ushort_as_half(r)); }
    static __device__ __forceinline__ T put(float u) { return __half_as_ushort(__float2half_rn(u)); }
    static __device__ __forceinline__ T bload(__amdgpu_buffer_rsrc_t b, unsigned v, unsigned s) {
        return __builtin_amdgcn_raw_buffer_load_b16(b, (int)v, (int)s, 0);
    }
    static __device__ __forceinline__ void bstore(__amdgpu_buffer_rsrc_t b, T q, unsigned v, unsigned s) {
        __builtin_amdgcn_raw_buffer_store_b16(q, b, (int)v, (int)s, 0);
    }
};
template <>
struct Raw<BF16> {
    typedef unsigned short T;
    static __device__ __forceinline__ float getu(T r) { return __uint_as_float((unsigned)r << 16); }
    static __device__ __forceinline__ T put(float u) { return __bfloat16_as_ushort(__float2bfloat16(u)); }
    static __device__ __forceinline__ T bload(__amdgpu_buffer_rsrc_t b, unsigned v, unsigned s) {
        return __builtin_amdgcn_raw_buffer_load_b16(b, (int)v, (int)s, 0);
    }
    static __device__ __forceinline__ void bstore(__amdgpu_buffer_rsrc_t b, T q, unsigned v, unsigned s) {
        __builtin_amdgcn_raw_buffer_store_b16(q, b, (int)v, (int)s, 0);
    }
};
template <>
struct Raw<SN16> {
    typedef short T;
    static __device__ __forceinline__ float getu(T r) { return sn16u_to_f(r); }
    static __device__ __forceinline__ T put(float u) { return f_to_sn16u(u); }
    static __device__ __forceinline__ T bload(__amdgpu_buffer_rsrc_t b, unsigned v, unsigned s) {
        return (short)__builtin_amdgcn_raw_buffer_load_b16(b, (int)v, (int)s, 0);
    }
    static __device__ __forceinline__ void bstore(__amdgpu_buffer_rsrc_t b, T q, unsigned v, unsigned s) {
        __builtin_amdgcn_raw_buffer_store_b16((unsigned short)q, b, (int)v, (int)s, 0);
    }
};

// Whether the intermediate iterate of a launch is rounded to the
// storage format: yes for the reference's SNORM16 format, which stores every
// iterate; the FP16/BF16 precision forms keep it in float.
template <class S>
struct RoundMid {
    static constexpr bool value = false;
};
template <>
struct RoundMid<SN16> {
    static constexpr bool value = true;
};

// Whether values in storage units differ from the values (m2 = |f|^2 then
// needs the factor 1/unit^2): all but F32.
template <class S>
struct UnitScaled {
    static constexpr bool value = true;
};
template <>
struct UnitScaled<F32> {
    static constexpr bool value = false;
};

__device__ __forceinline__ float lane_left(float v) {  // lane l gets lane l-1's value, lane 0 gets 0
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_right(float v) {  // lane l gets lane l+1's value, lane 63 gets 0
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}

template <class S>
struct ColsArgs {
    const typename S::T* f[3];
    const typename S::T* v[3];
    typename S::T* o[4];
    typename S::T* mid[3];  // MIDS: iterates 1 .. K-1, each three component volumes of n elements
    i64 n;
    Dims d;
    float mu, m2s, unit;
    int zc;
};

constexpr int NOT_VALU = 0x3fc;  // sched_barrier mask: all but vector arithmetic may move across
constexpr unsigned NO_LANE = 0x80000000u;  // a byte offset past every buffer resource: no memory access

template <class S, int K, int R, int NW, bool FINISH, bool MIDS>
struct Cols {
    typedef Raw<S> Q;
    typedef typename Q::T RT;
    static constexpr int ROWS = NW * R, OW = 64 - 2 * K, OH = ROWS - 2 * (K - 1);
    static constexpr int PR = R > 1 ? 2 : 1;  // published rows per wave
    struct Lds {
        float row[K][3][NW][PR][64];  // a wave's first and last row of every iterate
        float ring[3][3][64];         // iterate 0: the rows above and below the tile; not read
    };

    const ColsArgs<S>& a;
    Lds* L;
    int lane, w, row0, qs, qe, zb;
    int ledge, redge, yfix, yface;  // 0 or 1, uniform
    bool col0, colN;
    unsigned pb, rb, voff, hoff;
    unsigned svoff[R];  // store offset of the thread's lane, NO_LANE on rows it does not store
    unsigned ro[R];     // row offsets (uniform)
    // LDS words (within one buffer's row / ring arrays) of this wave and its y neighbours
    int pub, pdn, pup, pdn0, pup0, pring;
    __amdgpu_buffer_rsrc_t rv[3], rf[3], rs[4];

    // iterate 0 and f by plane modulo the ring, as stored; an F32 plane stays
    // in the registers it was loaded into until its last use
    RT v0[4][R][3], fr[4][R][3], hr[2][3];
    float P[K][R][3], C[K][R][3], fd[K][R][3];

    __device__ __forceinline__ Cols(const ColsArgs<S>& args, Lds* lds) : a(args), L(lds) {}

    __device__ __forceinline__ unsigned zoff(int z) const { return (unsigned)(clampi(z, 0, a.d.Z - 1) - zb) * pb; }

    __device__ __forceinline__ void load_v(RT (&q)[R][3], int z) {
        const unsigned sz = zoff(z);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) q[r][c] = Q::bload(rv[c], voff, sz + ro[r]);
    }
    __device__ __forceinline__ void load_f(RT (&q)[R][3], int z) {
        const unsigned sz = zoff(z);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) q[r][c] = Q::bload(rf[c], voff, sz + ro[r]);
    }
    __device__ __forceinline__ void load_ring(RT (&q)[3], int z) {
#pragma unroll
        for (int c = 0; c < 3; c++) q[c] = Q::bload(rv[c], hoff, zoff(z));
    }

    // this wave's published rows of a new plane of iterate k
    __device__ __forceinline__ void publish(int b, int k, const float (&v)[R][3]) {
        float* p = &L[b].row[k][0][0][0][0] + pub;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            p[c * (NW * PR * 64)] = v[0][c];
            if (PR == 2) p[c * (NW * PR * 64) + 64] = v[R - 1][c];
        }
    }
    __device__ __forceinline__ void publish_ring(int b, const RT (&h)[3]) {
#pragma unroll
        for (int c = 0; c < 3; c++) (&L[b].row[0][0][0][0][0])[pring + c * 192] = Q::getu(h[c]);
    }

    __device__ __forceinline__ void put_plane(const __amdgpu_buffer_rsrc_t* o, int nc, const RT (&q)[R][4],
                                              unsigned zo, unsigned mask) {
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (c < nc) Q::bstore(o[c], q[r][c], svoff[r] | mask, zo + ro[r]);
    }
    __device__ __forceinline__ void put_yfaces(const __amdgpu_buffer_rsrc_t* o, int nc, const RT (&q)[R][4],
                                               unsigned zo) {
        if (yface == 0) return;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int cy = row0 + r;
            if (cy == 2)
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (c < nc) Q::bstore(o[c], q[r][c], svoff[r], zo);
            if (cy == a.d.Y - 3)
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (c < nc) Q::bstore(o[c], q[r][c], svoff[r], zo + (unsigned)(a.d.Y - 1) * rb);
        }
    }
    // plane p of an iterate (its faces included) if this chunk stores it
    __device__ __forceinline__ void store(const __amdgpu_buffer_rsrc_t* o, bool with_w, int p, const float (&v)[R][3]) {
        RT q[R][4];
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int c = 0; c < 3; c++) q[r][c] = Q::put(v[r][c]);
            if (with_w) {
                // magnitude of the stored (rounded) components, 1 (in units) where 0
                const float x = Q::getu(q[r][0]), y = Q::getu(q[r][1]), z = Q::getu(q[r][2]);
                const float l = sqrtf(x * x + y * y + z * z);
                q[r][3] = Q::put(l > 0.0f ? l : a.unit);
            }
        }
        const int nc = with_w ? 4 : 3;
        const bool in = p >= qs && p < qe;
        const unsigned zo = zoff(in ? p : qs);
        put_plane(o, nc, q, zo, in ? 0u : NO_LANE);
        if (in && (yface != 0 || p == 2 || p == a.d.Z - 3)) {
            put_yfaces(o, nc, q, zo);
            if (p == 2) {
                put_plane(o, nc, q, zoff(0), 0u);
                put_yfaces(o, nc, q, zoff(0));
            }
            if (p == a.d.Z - 3) {
                put_plane(o, nc, q, zoff(a.d.Z - 1), 0u);
                put_yfaces(o, nc, q, zoff(a.d.Z - 1));
            }
        }
    }

    // the boundary lanes take the value two lanes over (column 0 from column 2)
    template <bool FIRST>
    __device__ __forceinline__ void from_mirror(float (&o)[R][3]) {
        float m[R][3];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) m[r][c] = FIRST ? lane_right(o[r][c]) : lane_left(o[r][c]);
        __builtin_amdgcn_sched_barrier(NOT_VALU);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) m[r][c] = FIRST ? lane_right(m[r][c]) : lane_left(m[r][c]);
        __builtin_amdgcn_sched_barrier(NOT_VALU);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) o[r][c] = (FIRST ? col0 : colN) ? m[r][c] : o[r][c];
    }

    // iterate k's rows below and above the thread's rows, from buffer b
    template <int b>
    __device__ __forceinline__ void neighbours(int k, float (&dn)[3], float (&up)[3]) {
        const float* p0 = &L[b].row[0][0][0][0][0];
        const float* p = &L[b].row[k][0][0][0][0];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            dn[c] = k == 0 ? p0[pdn0 + c * (w == 0 ? 192 : NW * PR * 64)] : p[pdn + c * (NW * PR * 64)];
            up[c] = k == 0 ? p0[pup0 + c * (w == NW - 1 ? 192 : NW * PR * 64)] : p[pup + c * (NW * PR * 64)];
        }
    }

    template <int U>
    __device__ __forceinline__ void step(int t) {
        constexpr int bw = U & 1, br = bw ^ 1;
        // y neighbours of the thread's first and last row
        float dn[3], up[3];
        neighbours<br>(0, dn, up);
        // the planes that arrive: iterate 0 of plane t + 1, f of plane t
        float N[R][3];
#pragma unroll
        for (int k = K - 1; k >= 1; k--)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < 3; c++) fd[k][r][c] = fd[k - 1][r][c];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                N[r][c] = Q::getu(v0[(U + 1) & 3][r][c]);
                fd[0][r][c] = Q::getu(fr[U & 3][r][c]);
            }
        publish(bw, 0, N);
        publish_ring(bw, hr[U & 1]);
        const bool zedge = t <= K || t >= a.d.Z - 2;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int p = t - k;
            if (k > 0 && zedge) {
                if (p == 1)
#pragma unroll
                    for (int r = 0; r < R; r++)
#pragma unroll
                        for (int c = 0; c < 3; c++) P[k][r][c] = N[r][c];
                if (p == a.d.Z - 2)
#pragma unroll
                    for (int r = 0; r < R; r++)
#pragma unroll
                        for (int c = 0; c < 3; c++) N[r][c] = P[k][r][c];
            }
            // in three rounds over the values: an instruction with a DPP operand
            // must not follow within two of one that writes a register it reads
            float s[R][3];
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < 3; c++) s[r][c] = -6.0f * C[k][r][c];
            __builtin_amdgcn_sched_barrier(NOT_VALU);
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < 3; c++) s[r][c] = s[r][c] + lane_right(C[k][r][c]);
            __builtin_amdgcn_sched_barrier(NOT_VALU);
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < 3; c++) s[r][c] = s[r][c] + lane_left(C[k][r][c]);
            __builtin_amdgcn_sched_barrier(NOT_VALU);
            if (k > 0) neighbours<br>(k, dn, up);
            if (k > 0 && yfix != 0) {
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        const int cy = row0 + r;
                        const float yp = r < R - 1 ? C[k][r < R - 1 ? r + 1 : r][c] : up[c];
                        const float ym = r > 0 ? C[k][r > 0 ? r - 1 : 0][c] : dn[c];
                        s[r][c] = s[r][c] + (cy == a.d.Y - 2 ? ym : yp);
                        s[r][c] = s[r][c] + (cy == 1 ? yp : ym);
                    }
            } else {
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        const float yp = r < R - 1 ? C[k][r < R - 1 ? r + 1 : r][c] : up[c];
                        const float ym = r > 0 ? C[k][r > 0 ? r - 1 : 0][c] : dn[c];
                        s[r][c] = s[r][c] + yp;
                        s[r][c] = s[r][c] + ym;
                    }
            }
            float o[R][3];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float* ff = fd[k][r];
                float m2 = ff[0] * ff[0] + ff[1] * ff[1] + ff[2] * ff[2];
                if (UnitScaled<S>::value) m2 = m2 * a.m2s;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    float l = s[r][c] + N[r][c];
                    l = l + P[k][r][c];
                    const float x = C[k][r][c] + (a.mu * l - (C[k][r][c] - ff[c]) * m2);
                    o[r][c] = RoundMid<S>::value && k < K - 1 ? Q::getu(Q::put(x)) : x;
                }
            }
            if (ledge + redge != 0) {
                if (ledge != 0)
                    from_mirror<true>(o);
                if (redge != 0)
                    from_mirror<false>(o);
            }
            if (k < K - 1) publish(bw, k + 1, o);
            if (MIDS && k < K - 1) {
                __amdgpu_buffer_rsrc_t om[3];
#pragma unroll
                for (int c = 0; c < 3; c++) om[c] = resource(a.mid[k] + c * a.n);
                store(om, false, p, o);
            }
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    P[k][r][c] = C[k][r][c];
                    C[k][r][c] = N[r][c];
                    N[r][c] = o[r][c];
                }
            // the plane below is free once stage 0 has used it
            if (k == 0) {
                load_v(v0[(U + 3) & 3], t + 3);
                load_ring(hr[U & 1], t + 3);
            }
        }
        load_f(fr[(U + 2) & 3], t + 2);
        store(rs, FINISH, t - (K - 1), N);
        __syncthreads();
    }

    // planes zb .. of a plane volume: those the chunk reads, and plane Z-1
    // when the chunk stores it.  The words are opaque so that every resource
    // keeps its own registers instead of being put together at each use.
    template <class T>
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(T* p) const {
        const int zspan = min(a.d.Z, qe + (K > 2 ? K : 2)) - zb;
        int n = __builtin_amdgcn_readfirstlane((int)(zspan * pb)), f = BUFFER_WORD3;
        asm volatile("" : "+s"(n), "+s"(f));
        return __builtin_amdgcn_make_buffer_rsrc((void*)(p + (i64)zb * a.d.X * a.d.Y), 0, n, f);
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
        const int ex = max(min(tbx * OW, d.X - 64), 0), ey = max(min(tby * OH, d.Y - ROWS), 0);
        const int cx = ex + lane;
        row0 = ey + w * R;
        qs = 1 + tbz * a.zc;
        qe = min(qs + a.zc, d.Z - 1);
        const int t0 = qs - (K - 1), te = qe + K - 2;
        zb = max(t0 - 1, 0);
        rb = (unsigned)d.X * (unsigned)sizeof(typename S::T);
        pb = rb * (unsigned)d.Y;
        voff = (unsigned)clampi(cx, 0, d.X - 1) * (unsigned)sizeof(typename S::T);
        hoff = NO_LANE;
        if (w == 0) hoff = voff + (unsigned)clampi(ey - 1, 0, d.Y - 1) * rb;
        if (w == NW - 1) hoff = voff + (unsigned)clampi(ey + ROWS, 0, d.Y - 1) * rb;
        col0 = cx == 0;
        colN = cx == d.X - 1;
        const int ring = K * 3 * NW * PR * 64;  // LDS words before Lds::ring
        pub = w * PR * 64 + lane;
        pdn = (w - (w > 0 ? 1 : 0)) * PR * 64 + (PR - 1) * 64 + lane;
        pup = (w + (w < NW - 1 ? 1 : 0)) * PR * 64 + lane;
        pdn0 = w == 0 ? ring + lane : pdn;
        pup0 = w == NW - 1 ? ring + 64 + lane : pup;
        pring = ring + (w == 0 ? 0 : (w == NW - 1 ? 64 : 128)) + lane;
        ledge = __builtin_amdgcn_readfirstlane(ex == 0);
        redge = __builtin_amdgcn_readfirstlane(ex + 63 >= d.X - 1);
        bool fix = false, face = false;
        const bool lane_out = (lane >= K || ex == 0) && (lane < 64 - K || ex + 64 >= d.X) && cx < d.X;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int j = w * R + r, cy = row0 + r;
            ro[r] = (unsigned)clampi(cy, 0, d.Y - 1) * rb;
            const bool out = (j >= K - 1 || ey == 0) && (j < ROWS - (K - 1) || ey + ROWS >= d.Y) && cy >= 1 && cy <= d.Y - 2;
            svoff[r] = out && lane_out ? voff : NO_LANE;
            fix = fix || cy == 1 || cy == d.Y - 2;
            face = face || (out && (cy == 2 || cy == d.Y - 3));
        }
        yfix = __builtin_amdgcn_readfirstlane(fix);
        yface = __builtin_amdgcn_readfirstlane(face);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            rv[c] = resource(a.v[c]);
            rf[c] = resource(a.f[c]);
            rs[c] = resource(a.o[c]);
        }
        if (FINISH) rs[3] = resource(a.o[3]);
        // the planes in flight at step t0: v t0-1 .. t0+2, f t0, t0+1 and the
        // ring rows of t0 .. t0+2
        {
            RT qh[3];
#pragma unroll
            for (int i = 0; i < 4; i++) load_v(v0[(i + 3) & 3], t0 - 1 + i);
            load_ring(qh, t0);
            load_ring(hr[0], t0 + 1);
            load_ring(hr[1], t0 + 2);
            load_f(fr[0], t0);
            load_f(fr[1], t0 + 1);
#pragma unroll
            for (int k = 0; k < K; k++)
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        P[k][r][c] = k == 0 ? Q::getu(v0[3][r][c]) : 0.0f;
                        C[k][r][c] = k == 0 ? Q::getu(v0[0][r][c]) : 0.0f;
                        fd[k][r][c] = 0.0f;
                    }
            publish(1, 0, C[0]);
            publish_ring(1, qh);
            __syncthreads();
        }
        // four steps per round, so that registers need no moves; up to three
        // past te, which store nothing (an exit after each step instead costs
        // 25 registers and makes the 16-bit forms spill)
        for (int t = t0; t <= te; t += 4) {
            step<0>(t);
            step<1>(t + 1);
            step<2>(t + 2);
            step<3>(t + 3);
        }
    }
};

template <class S, int K, int R, int NW, int WPE, bool FINISH, bool MIDS>
__global__ void __launch_bounds__(64 * NW, WPE) k_gvf_cols(ColsArgs<S> a) {
    typedef Cols<S, K, R, NW, FINISH, MIDS> M;
    __shared__ typename M::Lds lds[2];
    M m(a, lds);
    m.run();
}

// ---------------------------------------------------------------- host: form and chunk of a launch
// A built form of a marching kernel: K steps, R rows per wave, NW waves.
// occ: workgroups a CU holds; one, full: microseconds per step of one
// workgroup alone on a CU and of occ of them sharing it (measured at 4 to 136
// steps per launch, 64^3 to 512^3).
struct ColsForm {
    int K, R, NW, occ;
    float one, full;
};
inline dim3 cols_grid(const ColsForm& c, Dims d, int planes, int zc) {
    const int OW = 64 - 2 * c.K, rows = c.NW * c.R, OH = rows - 2 * (c.K - 1);
    return dim3(d.X > 64 ? (d.X - 64 + OW - 1) / OW + 1 : 1, d.Y > rows ? (d.Y - rows + OH - 1) / OH + 1 : 1,
                (planes + zc - 1) / zc);
}

// Planes per chunk of a form, and the estimated microseconds of a launch: a
// chunk of zc planes takes zc + 2 (K - 1) steps (rounded up to the loop's
// four), so short chunks repeat more steps and long ones leave CUs idle or a
// last round part full; a launch also moves `once` bytes a voxel and `halo`
// bytes that the planes beside a chunk repeat, and costs about 5 us to start
// and to fill the pipeline.  range: bytes per plane that a chunk's buffer
// resources cover (0: no limit from them).  max_blocks: workgroups that a
// launch may have.  us stays 1e30 where nothing fits.
struct ColsPlan {
    int form, zc;
    float us;
};
inline ColsPlan cols_plan(const ColsForm& c, int form, Dims d, int planes, double range, double halo, double once,
                          double max_blocks = 1e30) {
    const double cus = cu_count();
    ColsPlan best{form, 2, 1e30f};
    for (int steps = (2 * c.K + 3) & ~3; steps <= 140; steps += 4) {
        const int zc = steps - 2 * (c.K - 1);
        if (zc < 2 || range * (steps + 4) >= 2147483648.0) continue;
        const dim3 g = cols_grid(c, d, planes, zc);
        const double blocks = (double)g.x * g.y * g.z, per_cu = blocks / cus;
        double t;
        if (per_cu <= c.occ) {
            const double n = ceil(per_cu);
            t = c.occ > 1 ? c.one + (n - 1) * (c.full - c.one) / (c.occ - 1) : c.one;
        } else if (per_cu <= 4 * c.occ) {
            t = ceil(per_cu / c.occ - 0.5) * c.full + (per_cu / c.occ - floor(per_cu / c.occ) > 0.5 ? 0 : c.one);
        } else {
            t = (per_cu / c.occ + 0.5) * c.full;
        }
        const double memory = (double)d.n() * (halo * (zc + 2 * c.K) / zc + once) / 4.0e6;  // 4 TB/s
        const float us = (float)fmax(t * steps, memory) + 5.0f;
        if (us < best.us && blocks <= max_blocks) best = ColsPlan{form, zc, us};
        if (zc >= planes) break;
    }
    return best;
}

}  // namespace tsf
