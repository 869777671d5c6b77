// Segmentation from the centerline (segmentation.cpp:5-221, 223-307;
// kernels initGrowing, grow, dilate, erode, sphereSegmentation,
// kernels_no_3d_write.cl:1100-1234, 1370-1412).
//
// Inverse-gradient region growing: every centerline voxel seeds a cube of
// candidates (half size round(radius / 2) clamped to 1..4); a candidate X is
// accepted when some neighbour Y, not yet accepted, with a larger field
// magnitude than X's, has its normalised field pointing (among Y's 26
// neighbour directions) most nearly at X -- and Y becomes a candidate.
// Candidates that find no such Y are dropped.  The grown mask is closed
// (3x3x3 dilation, then erosion).
//
// The reference writes the next state in place from many threads: a
// candidate's own verdict and its neighbours' nominations of it land on the
// same byte in an unspecified order.  Here one pass records the verdicts
// (accepted) and the nominations apart and a second pass merges them with a
// fixed precedence, accepted > nominated > dropped: accepted voxels stay
// accepted and every pass that grows accepts a new voxel, so the iteration
// ends (as in the reference: at least two passes, then until a pass grows
// nothing).  The dilation starts from an empty volume (the image path
// initialises it; the buffer path leaves it uninitialised).
//
// Candidates are few, so a pass works on a list of them (k_seg_grow_list and
// k_seg_merge_list) and never reads the volume; passes are launched several
// at a time, each ending at once when the one before it grew nothing, and the
// host looks in after each batch.  300 x 288 x 320, 10 passes: 87 us a pass
// and a host round trip over the volume, 31 us without one on lists, most of
// it the scattered reads of the candidates' neighbours.  Volumes whose
// candidates fill more than a quarter of it overflow the lists and take the
// dense passes (k_seg_decide, k_seg_merge) from the start.
#include "field.hpp"

namespace tsf {

__device__ __forceinline__ bool inside(const Dims& d, int x, int y, int z) {
    return x >= 0 && y >= 0 && z >= 0 && x < d.X && y < d.Y && z < d.Z;
}
// clamp-to-edge read (the reference's image sampler)
__device__ __forceinline__ i64 clamped(const Dims& d, int x, int y, int z) {
    return d.at(clampi(x, 0, d.X - 1), clampi(y, 0, d.Y - 1), clampi(z, 0, d.Z - 1));
}

#define FOR_VOXEL(d)                                                              \
    const int x = blockIdx.x * 64 + threadIdx.x, y = blockIdx.y * 4 + threadIdx.y; \
    const int z = blockIdx.z;                                                     \
    if (x >= d.X || y >= d.Y) return;                                             \
    const i64 i = d.at(x, y, z);

// initGrowing: `out` holds a copy of the centerline; the seeds become 2.  A
// workgroup scans SEED_N voxels (16 a thread and access when the array allows)
// for centerline voxels, which are few, and its waves write their cubes.
// 300 x 288 x 320: 172 us with a thread per voxel, 24 us so.
constexpr int SEED_N = 4096;
template <bool VEC>
__global__ void __launch_bounds__(256) k_seg_seed(const uint8_t* __restrict__ cl, const float* __restrict__ radius,
                                                  uint8_t* out, Dims d) {
    __shared__ int list[SEED_N];
    __shared__ int n;
    if (threadIdx.x == 0) n = 0;
    __syncthreads();
    const i64 base = (i64)blockIdx.x * SEED_N, N = d.n();
    const int t0 = threadIdx.x * 16;
    if (VEC && base + t0 + 16 <= N) {
        const uint4 q = *reinterpret_cast<const uint4*>(cl + base + t0);
        const unsigned w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (w[k])
                for (int j = 0; j < 4; j++)
                    if (((w[k] >> (8 * j)) & 0xffu) == 1u) list[atomicAdd(&n, 1)] = t0 + 4 * k + j;
    } else {
        for (int j = 0; j < 16; j++)
            if (base + t0 + j < N && cl[base + t0 + j] == 1) list[atomicAdd(&n, 1)] = t0 + j;
    }
    __syncthreads();
    for (int k = threadIdx.x >> 6; k < n; k += 4) {
        const i64 i = base + list[k];
        const int x = (int)(i % d.X), y = (int)((i / d.X) % d.Y), z = (int)(i / ((i64)d.X * d.Y));
        const int H = min(max(1, (int)roundf(radius[i] / 2.0f)), 4), w = 2 * H + 1;
        for (int j = threadIdx.x & 63; j < w * w * w; j += 64) {
            const int c = j / (w * w), r = j - c * (w * w), b = r / w, a = r - b * w;
            const int nx = x + a - H, ny = y + b - H, nz = z + c - H;
            if (inside(d, nx, ny, nz) && cl[d.at(nx, ny, nz)] == 0) out[d.at(nx, ny, nz)] = 2;
        }
    }
}

// Whether the field (fx, fy, fz) points most nearly in direction (ta, tb, tc)
// of the 26: v = f . direction exceeds that of every direction before it in
// loop order and is not exceeded by one after it.  A NaN never wins.
__device__ __forceinline__ bool points_to(float fx, float fy, float fz, int ta, int tb, int tc) {
    const int kt = (ta + 1) * 9 + (tb + 1) * 3 + tc + 1;
    const float a = fabsf(fx), b = fabsf(fy), c = fabsf(fz), sum = a + b + c;
    if (sum >= 1e-30f && sum <= 1e30f) {
        // Only the seven directions with f's own signs can win: against a
        // sign leaving the component out gains at least 1.22 times, so does
        // it where the component is zero.  Signs do not alter a rounding.
        // (All 26 in turn made a grow pass 21 us for 17.)
        if (fx * ta < 0.0f || fy * tb < 0.0f || fz * tc < 0.0f) return false;
        const float u2 = 1.0f / sqrtf(2.0f), u3 = 1.0f / sqrtf(3.0f);
        const float v2x = a * u2, v2y = b * u2, v2z = c * u2;
        const float vxy = v2x + v2y, vxz = v2x + v2z, vyz = v2y + v2z, vxyz = (a * u3 + b * u3) + c * u3;
        const float vt = ta ? (tb ? (tc ? vxyz : vxy) : (tc ? vxz : a)) : (tb ? (tc ? vyz : b) : c);
        const int kx = fx < 0.0f ? -9 : 9, ky = fy < 0.0f ? -3 : 3, kz = fz < 0.0f ? -1 : 1;
        auto beaten = [&](float v, int k) { return 13 + k < kt ? v >= vt : v > vt; };
        return !(beaten(a, kx) || beaten(b, ky) || beaten(c, kz) || beaten(vxy, kx + ky) || beaten(vxz, kx + kz) ||
                 beaten(vyz, ky + kz) || beaten(vxyz, kx + ky + kz));
    }
    const float lt = sqrtf((float)(ta * ta + tb * tb + tc * tc));
    const float vt = fx * ((float)ta / lt) + fy * ((float)tb / lt) + fz * ((float)tc / lt);
    if (!(vt > -2.0f)) return false;
    for (int da = -1; da < 2; da++)
        for (int db = -1; db < 2; db++)
            for (int dc = -1; dc < 2; dc++) {
                const int k = (da + 1) * 9 + (db + 1) * 3 + dc + 1;
                if (k == 13 || k == kt) continue;
                const float l = sqrtf((float)(da * da + db * db + dc * dc));
                const float v = fx * ((float)da / l) + fy * ((float)db / l) + fz * ((float)dc / l);
                if (k < kt ? v >= vt : v > vt) return false;
            }
    return true;
}

// The neighbour (a, b, c) of candidate X: whether X is accepted by it (its
// voxel is then nominated).  wx = |F| at X; i the neighbour's index.
template <class S>
__device__ __forceinline__ bool accepted_by(const uint8_t* __restrict__ cur, const Field<S>& F, const Dims& d, int x,
                                            int y, int z, float wx, int a, int b, int c, i64& i) {
    i = clamped(d, x + a, y + b, z + c);
    const uint8_t state = cur[i];
    const float wy = F.mag(i);
    if (state == 1 || !(wy > wx) || !inside(d, x + a, y + b, z + c)) return false;
    return points_to(F.c(0, i) / wy, F.c(1, i) / wy, F.c(2, i) / wy, -a, -b, -c);
}

// grow, first half: the verdicts of the candidates and their nominations
template <class S>
__device__ __forceinline__ void decide_voxel(const uint8_t* __restrict__ cur, const Field<S>& F, const Dims& d, int x,
                                             int y, int z, i64 i, uint8_t* __restrict__ acc, uint8_t* nom,
                                             int32_t* grew) {
    const float wx = F.mag(i);
    bool cont = false;
    for (int a = -1; a < 2; a++)
        for (int b = -1; b < 2; b++)
            for (int c = -1; c < 2; c++) {
                if (a == 0 && b == 0 && c == 0) continue;
                i64 j;
                if (accepted_by<S>(cur, F, d, x, y, z, wx, a, b, c, j)) {
                    nom[j] = 1;
                    cont = true;
                }
            }
    if (cont) {
        acc[i] = 1;
        *grew = 1;
    }
}

// ---- growing on lists.  The marks of a voxel are bits of one byte, accepted
// and nominated for even and for odd passes: pass p sets those of its parity,
// its merge reads them, and the next merge clears the nominations (of the
// voxels that are its candidates); an accepted voxel never is a candidate
// again, so its mark may stay.  Slots: what pass p of a batch needs to know.
constexpr int SEG_BATCH = 8;
struct SegSlots {
    int32_t count[SEG_BATCH + 1];  // candidates of pass p (count[0] of the batch: carried over)
    int32_t grew[SEG_BATCH + 1];   // grew[p + 1]: pass p accepted a voxel; grew[0]: the pass before the batch
    int32_t overflow;
};
__device__ __forceinline__ bool seg_skip(const SegSlots* s, int p, bool first) {
    // the first two passes of all always run
    return s->overflow != 0 || (!(first && p < 2) && s->grew[p] == 0);
}
__device__ __forceinline__ unsigned mark(uint8_t* marks, i64 i, unsigned bit) {
    unsigned* w = reinterpret_cast<unsigned*>(marks) + (i >> 2);
    const int s = 8 * (int)(i & 3);
    return (atomicOr(w, bit << s) >> s) & 0xffu;
}

// 1 = begin a batch (the last one's end becomes slot 0), 0 = begin at all
__global__ void k_seg_begin(SegSlots* s, int next) {
    const int c = next ? s->count[SEG_BATCH] : 0, g = next ? s->grew[SEG_BATCH] : 0;
    for (int k = 0; k <= SEG_BATCH; k++) s->count[k] = s->grew[k] = 0;
    s->count[0] = c;
    s->grew[0] = g;
    if (!next) s->overflow = 0;
}

// Appends a workgroup's `n` entries to a list: one atomic on its counter.
// (An atomic per entry serialises on that one address: a grow pass at
// 300 x 288 x 320 took 151 us on average, 21 us with this.)
__device__ __forceinline__ void append(const int32_t* own, int n, int32_t* __restrict__ list, int cap, int32_t* count,
                                       int32_t* overflow) {
    __shared__ int base;
    if (threadIdx.x == 0) {
        base = n ? atomicAdd(count, n) : 0;
        if (base > cap - n) *overflow = 1;
    }
    __syncthreads();
    if (base <= cap - n)
        for (int k = threadIdx.x; k < n; k += blockDim.x) list[base + k] = own[k];
    __syncthreads();
}

// the list of voxels of value 2 (16 a thread; the padding is not counted)
__global__ void __launch_bounds__(256) k_seg_collect(const uint8_t* __restrict__ a, i64 n, int32_t* __restrict__ list,
                                                     int cap, SegSlots* s) {
    __shared__ int32_t own[4096];
    __shared__ int found;
    if (threadIdx.x == 0) found = 0;
    __syncthreads();
    const i64 t = 16 * ((i64)blockIdx.x * 256 + threadIdx.x);
    if (t < n) {
        const uint4 q = *reinterpret_cast<const uint4*>(a + t);  // a is a workspace array, padded to 256
        const unsigned w[4] = {q.x, q.y, q.z, q.w};
        unsigned hit = 0;
#pragma unroll
        for (int k = 0; k < 16; k++)
            if (((w[k >> 2] >> (8 * (k & 3))) & 0xffu) == 2u && t + k < n) hit |= 1u << k;
        if (hit) {
            int at = atomicAdd(&found, __popc(hit));
            for (int k = 0; k < 16; k++)
                if (hit & (1u << k)) own[at++] = (int32_t)(t + k);
        }
    }
    __syncthreads();
    if (found) append(own, found, list, cap, &s->count[0], &s->overflow);
}

// pass p, first half: the candidates of `list` (those still 2), the voxels
// they nominate appended to `next` once each.  32 threads per candidate, a
// neighbour each.
constexpr int GROW_OWN = 2048;  // nominations a workgroup holds back
template <class S>
__global__ void __launch_bounds__(256) k_seg_grow_list(const uint8_t* __restrict__ cur, Field<S> F, Dims d,
                                                       const int32_t* __restrict__ list, int32_t* __restrict__ next,
                                                       int cap, uint8_t* marks, SegSlots* s, int p, bool first) {
    __shared__ int32_t own[GROW_OWN];
    __shared__ int found, grown, skip;
    // One verdict for the workgroup: another one's append may set the overflow
    // mark at any time, and waves that read it apart would part ways here.
    if (threadIdx.x == 0) {
        skip = seg_skip(s, p, first);
        found = grown = 0;
    }
    __syncthreads();
    if (skip) return;
    const unsigned accepted = (p & 1) ? 4u : 1u, nominated = 2 * accepted;
    const int count = s->count[p];
    const int sub = threadIdx.x & 31;
    const int a = sub / 9 - 1, b = sub / 3 % 3 - 1, c = sub % 3 - 1;
    for (int k0 = blockIdx.x * 8; k0 < count; k0 += gridDim.x * 8) {
        const int k = k0 + (threadIdx.x >> 5);
        bool yes = false;
        i64 i = 0;
        if (k < count) {
            const int ii = list[k];
            i = ii;
            const uint8_t state = cur[i];
            const float wx = F.mag(i);
            if (state == 2 && sub < 27 && sub != 13) {
                const int row = ii / d.X, x = ii - row * d.X, z = row / d.Y, y = row - z * d.Y;
                i64 j;
                yes = accepted_by<S>(cur, F, d, x, y, z, wx, a, b, c, j);
                if (yes && !(mark(marks, j, nominated) & nominated)) own[atomicAdd(&found, 1)] = (int32_t)j;
            }
        }
        const unsigned long long m = __ballot(yes);
        const unsigned any = (unsigned)((threadIdx.x & 32) ? m >> 32 : m);
        if (sub == 0 && any) {
            mark(marks, i, accepted);
            grown = 1;
        }
        __syncthreads();
        const int held = found;
        __syncthreads();
        if (held > GROW_OWN - 8 * 26) {
            append(own, held, next, cap, &s->count[p + 1], &s->overflow);
            if (threadIdx.x == 0) found = 0;
            __syncthreads();
        }
    }
    if (found) append(own, found, next, cap, &s->count[p + 1], &s->overflow);
    if (threadIdx.x == 0 && grown) s->grew[p + 1] = 1;
}

// pass p, second half: accepted > nominated > dropped on both lists
__global__ void __launch_bounds__(256) k_seg_merge_list(uint8_t* cur, const int32_t* __restrict__ list,
                                                        const int32_t* __restrict__ next, uint8_t* marks,
                                                        const SegSlots* s, int p, bool first) {
    if (seg_skip(s, p, first)) return;
    const unsigned accepted = (p & 1) ? 4u : 1u, nominated = 2 * accepted, old = (p & 1) ? 2u : 8u;
    const int count = s->count[p], noms = s->count[p + 1];
    for (int k = blockIdx.x * 256 + threadIdx.x; k < count + noms; k += gridDim.x * 256) {
        if (k < count) {
            const i64 i = list[k];
            unsigned* w = reinterpret_cast<unsigned*>(marks) + (i >> 2);
            const int sh = 8 * (int)(i & 3);
            const unsigned m = (atomicAnd(w, ~(old << sh)) >> sh) & 0xffu;
            if (cur[i] == 2) {
                if (m & accepted) cur[i] = 1;
                else if (!(m & nominated)) cur[i] = 0;
            }
        } else {
            const i64 i = next[k - count];
            const unsigned m = marks[i];
            cur[i] = cur[i] == 1 || (m & accepted) ? 1 : 2;
        }
    }
}

template <class S>
__global__ void k_seg_decide(const uint8_t* __restrict__ cur, Field<S> F, Dims d, uint8_t* __restrict__ acc,
                             uint8_t* nom, int32_t* grew) {
    FOR_VOXEL(d)
    if (cur[i] == 2) decide_voxel<S>(cur, F, d, x, y, z, i, acc, nom, grew);
}

// grow, second half: accepted > nominated > dropped; clears the marks.
// Elementwise over the 256-byte-aligned workspace arrays (their lengths are
// multiples of 256), 16 voxels per thread; the padding past the last voxel
// is merged too and never read as a voxel.
__device__ __forceinline__ unsigned merge_word(unsigned c, unsigned a, unsigned m) {
    unsigned o = 0;
#pragma unroll
    for (int k = 0; k < 32; k += 8) {
        const unsigned cb = (c >> k) & 0xffu, ab = (a >> k) & 0xffu, mb = (m >> k) & 0xffu;
        o |= (cb == 1u || ab ? 1u : (mb ? 2u : 0u)) << k;
    }
    return o;
}
__global__ void __launch_bounds__(256) k_seg_merge(const uint4* __restrict__ cur, uint4* __restrict__ acc,
                                                   uint4* __restrict__ nom, uint4* __restrict__ next, i64 n16) {
    const i64 t = (i64)blockIdx.x * 256 + threadIdx.x;
    if (t >= n16) return;
    const uint4 c = cur[t], a = acc[t], m = nom[t];
    next[t] = make_uint4(merge_word(c.x, a.x, m.x), merge_word(c.y, a.y, m.y), merge_word(c.z, a.z, m.z),
                         merge_word(c.w, a.w, m.w));
    acc[t] = make_uint4(0, 0, 0, 0);
    nom[t] = make_uint4(0, 0, 0, 0);
}

// The 3x3x3 closing, one axis per pass (a box is the product of its three
// axis ranges, and both the inside-the-volume test of the dilation and the
// clamp-to-edge of the erosion act per axis):
// dilate: 1 where a voxel of the axis neighbourhood inside the volume is 1;
template <int AXIS>
__global__ void k_seg_dilate_axis(const uint8_t* __restrict__ in, uint8_t* __restrict__ out, Dims d) {
    FOR_VOXEL(d)
    const int p = AXIS == 0 ? x : (AXIS == 1 ? y : z), e = AXIS == 0 ? d.X : (AXIS == 1 ? d.Y : d.Z);
    const i64 s = AXIS == 0 ? 1 : (AXIS == 1 ? (i64)d.X : (i64)d.X * d.Y);
    const bool v = in[i] == 1 || (p > 0 && in[i - s] == 1) || (p + 1 < e && in[i + s] == 1);
    out[i] = v ? 1 : 0;
}
// erode: 1 where the axis neighbourhood (clamp-to-edge) is all 1.
template <int AXIS>
__global__ void k_seg_erode_axis(const uint8_t* __restrict__ in, uint8_t* __restrict__ out, Dims d) {
    FOR_VOXEL(d)
    const int p = AXIS == 0 ? x : (AXIS == 1 ? y : z), e = AXIS == 0 ? d.X : (AXIS == 1 ? d.Y : d.Z);
    const i64 s = AXIS == 0 ? 1 : (AXIS == 1 ? (i64)d.X : (i64)d.X * d.Y);
    const bool v = in[i] == 1 && in[p > 0 ? i - s : i] == 1 && in[p + 1 < e ? i + s : i] == 1;
    out[i] = v ? 1 : 0;
}

// The same on 32-bit words (4 voxels along x) when X is a multiple of 4, so
// that no word crosses a row, all three axes in one pass: a thread marches a
// column of words in z, keeps the last two planes' x-y results and stores
// their combination with the new one.  Words of a plane go to lanes in index
// order, so a word's x neighbours are in the next lanes (the wave's ends load
// theirs).  Each byte of a word is taken as 1 where it is 1 and else 0; along
// x the neighbour bytes come from the adjacent words (little-endian: byte k
// is x0 + k), zero (dilation) or the edge byte itself (erosion) past the row
// ends, and rows and planes past the volume are zero or repeat the edge.
// 300 x 288 x 320: 147 us for the closing in six one-axis passes, 42 us
// in these two.
__device__ __forceinline__ unsigned is1(unsigned w) {
    const unsigned t = w ^ 0x01010101u;
    return (~(((t & 0x7f7f7f7fu) + 0x7f7f7f7fu) | t) >> 7) & 0x01010101u;
}
constexpr int CLOSE_ZC = 16;  // planes per workgroup of the word passes
// the rows around word q of a plane
template <bool DILATE>
__device__ __forceinline__ unsigned close_rows(const unsigned* __restrict__ in, int q, int up, int down) {
    const unsigned a = in[q], b = in[q + up], c = in[q + down];
    // the erosion's input is the dilation's result: zeros and ones
    return DILATE ? is1(a) | is1(b) | is1(c) : a & b & c;
}
template <bool DILATE>
__global__ void __launch_bounds__(256) k_seg_close_words(const unsigned* __restrict__ in, unsigned* __restrict__ out,
                                                         Dims d) {
    const int XW = d.X >> 2, PW = XW * d.Y;
    const int q0 = blockIdx.x * 256 + threadIdx.x, q = min(q0, PW - 1);
    const int xw = q % XW, y = q / XW, lane = threadIdx.x & 63;
    // rows past the volume: the row itself (it changes neither an OR nor an AND)
    const int up = y > 0 ? -XW : 0, down = y + 1 < d.Y ? XW : 0;
    const int z0 = blockIdx.y * CLOSE_ZC, z1 = min(d.Z, z0 + CLOSE_ZC);
    const bool first = xw == 0, last = xw + 1 == XW;
    auto plane = [&](int z) -> unsigned {
        const unsigned* in_z = in + (i64)PW * clampi(z, 0, d.Z - 1);
        const unsigned c = close_rows<DILATE>(in_z, q, up, down);
        unsigned lw = __shfl_up(c, 1), hw = __shfl_down(c, 1);
        if (lane == 0 && !first) lw = close_rows<DILATE>(in_z, q - 1, up, down);
        if (lane == 63 && !last) hw = close_rows<DILATE>(in_z, q + 1, up, down);
        const unsigned l = first ? (DILATE ? 0u : c & 0xffu) : lw >> 24;
        const unsigned h = last ? (DILATE ? 0u : c & 0xff000000u) : (hw & 0xffu) << 24;
        const unsigned left = (c << 8) | l, right = (c >> 8) | h;
        // planes past the volume repeat the edge's, which changes neither an OR nor an AND
        return DILATE ? (c | left | right) : (c & left & right);
    };
    unsigned below = plane(z0 - 1), here = plane(z0);
    for (int z = z0; z < z1; z++) {
        const unsigned above = plane(z + 1);
        if (q0 < PW) out[(i64)PW * z + q] = DILATE ? (below | here | above) : (below & here & above);
        below = here;
        here = above;
    }
}

// sphereSegmentation: a ball of the voxel's radius (|offset| < r) around
// every centerline voxel
__global__ void k_seg_spheres(const uint8_t* __restrict__ cl, const float* __restrict__ radius, uint8_t* out, Dims d) {
    FOR_VOXEL(d)
    if (cl[i] == 0) return;
    const float r = radius[i];
    const int N = (int)ceilf(r);
    for (int a = -N; a <= N; a++)
        for (int b = -N; b <= N; b++)
            for (int c = -N; c <= N; c++)
                if (sqrtf((float)a * (float)a + (float)b * (float)b + (float)c * (float)c) < r &&
                    inside(d, x + a, y + b, z + c))
                    out[d.at(x + a, y + b, z + c)] = 1;
}

template <class S>
static void launch_decide(const tsf_field* f, const uint8_t* cur, Dims d, uint8_t* acc, uint8_t* nom, int32_t* grew,
                          hipStream_t stream) {
    typedef typename S::T T;
    Field<S> F{(const T*)f->x, (const T*)f->y, (const T*)f->z, (const T*)f->w, 1.0f / f->scale};
    dim3 grid((d.X + 63) / 64, (d.Y + 3) / 4, d.Z), block(64, 4);
    hipLaunchKernelGGL(k_seg_decide<S>, grid, block, 0, stream, cur, F, d, acc, nom, grew);
}

template <class S>
static void launch_grow(const tsf_field* f, const uint8_t* cur, Dims d, const int32_t* list, int32_t* next, int cap,
                        uint8_t* marks, SegSlots* slots, int p, bool first, hipStream_t stream) {
    typedef typename S::T T;
    Field<S> F{(const T*)f->x, (const T*)f->y, (const T*)f->z, (const T*)f->w, 1.0f / f->scale};
    hipLaunchKernelGGL(k_seg_grow_list<S>, 1024, 256, 0, stream, cur, F, d, list, next, cap, marks, slots, p, first);
}

static void launch_seed(const uint8_t* cl, const float* radius, uint8_t* out, Dims d, hipStream_t stream) {
    const unsigned g = (unsigned)((d.n() + SEED_N - 1) / SEED_N);
    if ((uintptr_t)cl % 16 == 0) hipLaunchKernelGGL(k_seg_seed<true>, g, 256, 0, stream, cl, radius, out, d);
    else hipLaunchKernelGGL(k_seg_seed<false>, g, 256, 0, stream, cl, radius, out, d);
}

// Growing on lists: `cur` holds the centerline and its seeds; marks is clear.
// even, odd: lists of `cap` entries.  *passes = the passes run, or -1 when a list
// overflowed (cur is then part grown).
static tsf_status grow_on_lists(const tsf_field* f, uint8_t* cur, Dims d, int32_t* even, int32_t* odd, int cap,
                                uint8_t* marks, SegSlots* slots, i64* passes, hipStream_t stream, const char* W) {
    const i64 n = d.n();
    hipLaunchKernelGGL(k_seg_begin, 1, 1, 0, stream, slots, 0);
    hipLaunchKernelGGL(k_seg_collect, (unsigned)((n + 4095) / 4096), 256, 0, stream, cur, n, even, cap, slots);
    for (i64 done = 0;; done += SEG_BATCH) {
        const bool first = done == 0;
        if (!first) hipLaunchKernelGGL(k_seg_begin, 1, 1, 0, stream, slots, 1);
        for (int p = 0; p < SEG_BATCH; p++) {
            // SEG_BATCH is even: pass p of every batch reads the list of its parity
            int32_t *list = (p & 1) ? odd : even, *next = (p & 1) ? even : odd;
            switch (f->storage) {
                case TSF_STORAGE_F32: launch_grow<F32>(f, cur, d, list, next, cap, marks, slots, p, first, stream); break;
                case TSF_STORAGE_F16: launch_grow<F16>(f, cur, d, list, next, cap, marks, slots, p, first, stream); break;
                case TSF_STORAGE_SN16: launch_grow<SN16>(f, cur, d, list, next, cap, marks, slots, p, first, stream); break;
                default: launch_grow<BF16>(f, cur, d, list, next, cap, marks, slots, p, first, stream);
            }
            hipLaunchKernelGGL(k_seg_merge_list, 256, 256, 0, stream, cur, list, next, marks, slots, p, first);
        }
        TSF_TRY(check_launch(W));
        SegSlots h;
        hipError_t e = hipMemcpyAsync(&h, slots, sizeof h, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (e != hipSuccess) return set_error(TSF_ERR_HIP, "%s: %s", W, hipGetErrorString(e));
        if (h.overflow) {
            *passes = -1;
            return TSF_OK;
        }
        // the first pass after the first of all that grew nothing was the last
        for (int p = 0; p < SEG_BATCH; p++)
            if (!(first && p == 0) && (h.grew[p + 1] == 0 || done + p > n + 2)) {
                *passes = done + p + 1;
                return TSF_OK;
            }
    }
}

}  // namespace tsf

using namespace tsf;

extern "C" {

size_t tsf_segment_inverse_gradient_workspace_size(tsf_dims dims) {
    const size_t n = (size_t)D(dims).n();
    return 4 * ((n + 255) & ~(size_t)255) + 256;
}

tsf_status tsf_segment_inverse_gradient(const uint8_t* centerlines, const float* radius, const tsf_field* field,
                                        tsf_dims dims, uint8_t* segmentation, int32_t* iterations, void* workspace,
                                        size_t workspace_bytes, hipStream_t stream) {
    const char* W = "tsf_segment_inverse_gradient";
    if (!centerlines || !radius || !segmentation) return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: NULL argument", W);
    TSF_TRY(check_field(field, true, W));
    TSF_TRY(check_dims(dims, 1, W));
    Dims d = D(dims);
    const i64 n = d.n();
    Scratch sc;
    TSF_TRY(sc.get(workspace, workspace_bytes, tsf_segment_inverse_gradient_workspace_size(dims), W));
    const size_t nb = ((size_t)n + 255) & ~(size_t)255;
    uint8_t* A = (uint8_t*)sc.ptr;
    uint8_t* B = A + nb;
    uint8_t* acc = B + nb;
    uint8_t* nom = acc + nb;
    int32_t* grew = (int32_t*)(nom + nb);
    dim3 grid((d.X + 63) / 64, (d.Y + 3) / 4, d.Z), block(64, 4);
    hipError_t e = hipMemcpyAsync(A, centerlines, n, hipMemcpyDeviceToDevice, stream);
    if (e == hipSuccess) e = hipMemsetAsync(acc, 0, nb, stream);
    if (e != hipSuccess) return set_error(TSF_ERR_HIP, "%s: %s", W, hipGetErrorString(e));
    launch_seed(centerlines, radius, A, d, stream);
    TSF_TRY(check_launch(W));
    // at least two passes, then until a pass grows nothing; a pass that
    // grows accepts a new voxel, so there are at most n + 2 of them
    i64 passes = -1;
    if (n < ((i64)1 << 31))
        TSF_TRY(grow_on_lists(field, A, d, (int32_t*)B, (int32_t*)nom, (int)(nb / 4), acc, (SegSlots*)grew, &passes,
                              stream, W));
    if (passes < 0) {
        e = hipMemcpyAsync(A, centerlines, n, hipMemcpyDeviceToDevice, stream);
        if (e == hipSuccess) e = hipMemsetAsync(acc, 0, 2 * nb, stream);
        if (e != hipSuccess) return set_error(TSF_ERR_HIP, "%s: %s", W, hipGetErrorString(e));
        launch_seed(centerlines, radius, A, d, stream);
        TSF_TRY(check_launch(W));
        i64 pass = 0;
        for (;; pass++) {
            int32_t g = 0;
            e = hipMemsetAsync(grew, 0, sizeof(int32_t), stream);
            if (e != hipSuccess) return set_error(TSF_ERR_HIP, "%s: %s", W, hipGetErrorString(e));
            switch (field->storage) {
                case TSF_STORAGE_F32: launch_decide<F32>(field, A, d, acc, nom, grew, stream); break;
                case TSF_STORAGE_F16: launch_decide<F16>(field, A, d, acc, nom, grew, stream); break;
                case TSF_STORAGE_SN16: launch_decide<SN16>(field, A, d, acc, nom, grew, stream); break;
                default: launch_decide<BF16>(field, A, d, acc, nom, grew, stream);
            }
            hipLaunchKernelGGL(k_seg_merge, (unsigned)((nb / 16 + 255) / 256), 256, 0, stream, (const uint4*)A,
                               (uint4*)acc, (uint4*)nom, (uint4*)B, (i64)(nb / 16));
            TSF_TRY(check_launch(W));
            std::swap(A, B);
            if (pass == 0) continue;
            e = hipMemcpyAsync(&g, grew, sizeof g, hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipStreamSynchronize(stream);
            if (e != hipSuccess) return set_error(TSF_ERR_HIP, "%s: %s", W, hipGetErrorString(e));
            if (g == 0 || pass > n + 2) break;
        }
        passes = pass + 1;
    }
    if (iterations) *iterations = (int32_t)passes;
    // closing: A -> B (dilation) -> segmentation (erosion), or an axis a
    // pass: A -> acc -> nom -> B, B -> acc -> nom -> segmentation
    if (d.X % 4 == 0 && ((uintptr_t)segmentation & 3u) == 0 && (i64)d.X * d.Y < ((i64)1 << 31)) {
        const dim3 gw((unsigned)((i64)(d.X / 4) * d.Y + 255) / 256, (d.Z + CLOSE_ZC - 1) / CLOSE_ZC);
        hipLaunchKernelGGL(k_seg_close_words<true>, gw, 256, 0, stream, (const unsigned*)A, (unsigned*)B, d);
        hipLaunchKernelGGL(k_seg_close_words<false>, gw, 256, 0, stream, (const unsigned*)B,
                           (unsigned*)segmentation, d);
    } else {
        hipLaunchKernelGGL(k_seg_dilate_axis<0>, grid, block, 0, stream, A, acc, d);
        hipLaunchKernelGGL(k_seg_dilate_axis<1>, grid, block, 0, stream, acc, nom, d);
        hipLaunchKernelGGL(k_seg_dilate_axis<2>, grid, block, 0, stream, nom, B, d);
        hipLaunchKernelGGL(k_seg_erode_axis<0>, grid, block, 0, stream, B, acc, d);
        hipLaunchKernelGGL(k_seg_erode_axis<1>, grid, block, 0, stream, acc, nom, d);
        hipLaunchKernelGGL(k_seg_erode_axis<2>, grid, block, 0, stream, nom, segmentation, d);
    }
    TSF_TRY(check_launch(W));
    if (sc.owned) {
        e = hipStreamSynchronize(stream);
        if (e != hipSuccess) return set_error(TSF_ERR_HIP, "%s: %s", W, hipGetErrorString(e));
    }
    return TSF_OK;
}

tsf_status tsf_segment_spheres(const uint8_t* centerlines, const float* radius, tsf_dims dims, uint8_t* segmentation,
                               hipStream_t stream) {
    const char* W = "tsf_segment_spheres";
    if (!centerlines || !radius || !segmentation) return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: NULL argument", W);
    TSF_TRY(check_dims(dims, 1, W));
    Dims d = D(dims);
    hipError_t e = hipMemsetAsync(segmentation, 0, (size_t)d.n(), stream);
    if (e != hipSuccess) return set_error(TSF_ERR_HIP, "%s: %s", W, hipGetErrorString(e));
    dim3 grid((d.X + 63) / 64, (d.Y + 3) / 4, d.Z), block(64, 4);
    hipLaunchKernelGGL(k_seg_spheres, grid, block, 0, stream, centerlines, radius, segmentation, d);
    return check_launch(W);
}

}  // extern "C"
