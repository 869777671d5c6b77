// Hessian eigenanalysis, candidate non-maximum suppression and cube maximum.
// Gather/VALU-bound per-voxel kernels; the eigensolver runs in registers
// (eigen3.hpp).  The circle-fitting TDF lives in circle.hip.
#include "eigen3.hpp"
#include "field.hpp"

namespace tsf {

template <class S, bool NORM>
__global__ void __launch_bounds__(256) k_hessian_eigen(Field<S> F, Dims d, float* __restrict__ lam,
                                                       float* __restrict__ vec) {
    const int x = blockIdx.x * 64 + threadIdx.x, y = blockIdx.y * 4 + threadIdx.y, z = blockIdx.z;
    if (x >= d.X || y >= d.Y) return;
    float H[3][3], V[3][3], ev[3];
    hessian<NORM>(F, d, x, y, z, H);
    eigen3(H, V, ev);
    const i64 i = d.at(x, y, z), N = d.n();
    lam[i] = ev[0];
    lam[N + i] = ev[1];
    lam[2 * N + i] = ev[2];
    if (vec) {
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int k = 0; k < 3; k++) vec[(3 * j + k) * N + i] = V[k][j];
    }
}

// doEigen (eigenanalysisOfHessian.cpp:264-389): samples divided by the
// host-style magnitude sqrt(Fx^2+Fy^2+Fz^2) of their voxel; no clamping.
__global__ void k_do_eigen_points(const float* __restrict__ Fx, const float* __restrict__ Fy,
                                  const float* __restrict__ Fz, Dims d, const int32_t* __restrict__ pos, i64 count,
                                  float* __restrict__ out) {
    i64 t = blockIdx.x * (i64)blockDim.x + threadIdx.x;
    if (t >= count) return;
    const int x = pos[3 * t], y = pos[3 * t + 1], z = pos[3 * t + 2];
    float* o = out + 12 * t;
    if (x < 1 || y < 1 || z < 1 || x > d.X - 2 || y > d.Y - 2 || z > d.Z - 2) {
        // the reference reads outside the arrays here; report NaN instead
#pragma unroll
        for (int k = 0; k < 12; k++) o[k] = __builtin_nanf("");
        return;
    }
    auto nv = [&](const float* c, int xx, int yy, int zz) -> float {
        i64 i = d.at(xx, yy, zz);
        return c[i] / sqrtf(Fx[i] * Fx[i] + Fy[i] * Fy[i] + Fz[i] * Fz[i]);
    };
    const float fxx = 0.5f * (nv(Fx, x + 1, y, z) - nv(Fx, x - 1, y, z));
    const float fyx = 0.5f * (nv(Fy, x + 1, y, z) - nv(Fy, x - 1, y, z));
    const float fyy = 0.5f * (nv(Fy, x, y + 1, z) - nv(Fy, x, y - 1, z));
    const float fzx = 0.5f * (nv(Fz, x + 1, y, z) - nv(Fz, x - 1, y, z));
    const float fzy = 0.5f * (nv(Fz, x, y + 1, z) - nv(Fz, x, y - 1, z));
    const float fzz = 0.5f * (nv(Fz, x, y, z + 1) - nv(Fz, x, y, z - 1));
    float H[3][3] = {{fxx, fyx, fzx}, {fyx, fyy, fzy}, {fzx, fzy, fzz}};
    float V[3][3], ev[3];
    eigen3(H, V, ev);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        o[k] = ev[k];
        o[3 + k] = V[k][0];
        o[6 + k] = V[k][1];
        o[9 + k] = V[k][2];
    }
}

// findCandidateCenterpoints2, kernels_no_3d_write.cl:1019-1084: a candidate
// is rejected if a voxel at offset r, 0 < |r| < maxD, whose direction lies
// within 0.5 rad of the plane normal to e1, has a smaller magnitude.
//
// The angle test of the reference, theta = acos(r/|r| . p/|p|) with p = r -
// e1 (e1 . r), is sin^2 of the angle between r and that plane: for a unit e1
// theta < 0.5 where (e1 . r)^2 < sin^2(0.5) |r|^2.  Offsets clear of that
// bound by 1e-4 |r|^2 (the float expressions are within 1e-5 of it) are
// decided by it; the others, and all of them when e1 is not of unit length to
// 1e-5, by the reference's own expressions.  So are the two ends:
//   - r in the plane: the cosine may round to more than 1, its acos is NaN and
//     the offset does not count (36 of the 192 offsets across an axis-aligned
//     tube with |r| < 8).  Its rounding error is below 6e-7 (ten roundings), its
//     distance from 1 half of (e1 . r)^2 / |r|^2;
//   - r along e1: p is what rounding leaves and may point anywhere.
// (Evaluated for 1326 axes and all offsets up to 63, the expressions differ from
// the bound at and below 2.0e-7 and at and above 0.99999 of |r|^2 only.)  They
// are asked about darker voxels alone, of which a survivor has few.
struct NmsCandidate {
    int x, y, z, maxD;
    float ex, ey, ez, wp;
    bool unit;
};
template <class S>
__device__ __forceinline__ bool nms_beaten(const NmsCandidate& q, const Field<S>& F, const Dims& d, int a, int b,
                                           int c) {
    const int n2 = a * a + b * b + c * c;
    if (n2 == 0 || n2 >= q.maxD * q.maxD) return false;
    const float rx = (float)a, ry = (float)b, rz = (float)c;
    const float dp = q.ex * rx + q.ey * ry + q.ez * rz;
    const float r2 = (float)n2, d2 = dp * dp;
    if (q.unit && d2 > 0.2299488f * r2 && d2 < 0.999f * r2) return false;
    const int nx = clampi(q.x + a, 0, d.X - 1), ny = clampi(q.y + b, 0, d.Y - 1), nz = clampi(q.z + c, 0, d.Z - 1);
    if (!(F.mag(d.at(nx, ny, nz)) < q.wp)) return false;
    if (q.unit && d2 < 0.2297488f * r2 && d2 > 4e-6f * r2) return true;
    const float px = rx - q.ex * dp, py = ry - q.ey * dp, pz = rz - q.ez * dp;
    const float lr = sqrtf(rx * rx + ry * ry + rz * rz);
    const float lp = sqrtf(px * px + py * py + pz * pz);
    const float cs = (rx / lr) * (px / lp) + (ry / lr) * (py / lp) + (rz / lr) * (pz / lp);
    return acosf(cs) < 0.5f;
}
// A thread solves for its candidate's e1 and looks at the 26 voxels next to
// it, which rejects most candidates off the axis; the survivors with a wider
// reach are collected in LDS and a wave searches each of them, 64 offsets at
// a time.  192298 candidates of tubes up to radius 8 (reach up to 8: 4913
// offsets): 3267 us with a thread per candidate and the reference's
// expressions at every offset, 89 us so.
template <class S>
__global__ void __launch_bounds__(256) k_candidate_nms(const float* __restrict__ radius, Field<S> F, Dims d,
                                                       const int32_t* __restrict__ pos, i64 count, int cap,
                                                       uint8_t* __restrict__ out) {
    __shared__ NmsCandidate list[256];
    __shared__ int n;
    if (threadIdx.x == 0) n = 0;
    __syncthreads();
    const i64 t = blockIdx.x * (i64)blockDim.x + threadIdx.x;
    if (t < count) {
        NmsCandidate q;
        q.x = pos[3 * t];
        q.y = pos[3 * t + 1];
        q.z = pos[3 * t + 2];
        // a position that is not a voxel is ignored
        if (q.x >= 0 && q.y >= 0 && q.z >= 0 && q.x < d.X && q.y < d.Y && q.z < d.Z) {
            const i64 i = d.at(q.x, q.y, q.z);
            q.maxD = (int)fmaxf(fminf(roundf(radius[i]), (float)cap), 1.0f);
            bool valid = true;
            if (q.maxD > 1) {
                float H[3][3], V[3][3], ev[3];
                hessian<true>(F, d, q.x, q.y, q.z, H);
                eigen3(H, V, ev);
                q.ex = V[0][0];
                q.ey = V[1][0];
                q.ez = V[2][0];
                q.wp = F.mag(i);
                q.unit = fabsf(q.ex * q.ex + q.ey * q.ey + q.ez * q.ez - 1.0f) < 1e-5f;
                for (int c = -1; c <= 1; c++)
                    for (int b = -1; b <= 1; b++)
                        for (int a = -1; a <= 1; a++)
                            if (nms_beaten(q, F, d, a, b, c)) valid = false;
            }
            if (valid && q.maxD > 2) list[atomicAdd(&n, 1)] = q;
            else out[i] = valid;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    for (int k = threadIdx.x >> 6; k < n; k += 4) {
        const NmsCandidate q = list[k];
        const int m = q.maxD - 1, w = 2 * m + 1, total = w * w * w;  // |r| < maxD: components to maxD - 1
        bool beaten = false;
        for (int j = lane; j - lane < total && !beaten; j += 64) {
            const int c = j / (w * w), r = j - c * (w * w), b = r / w, a = r - b * w;
            beaten = __any(j < total && nms_beaten(q, F, d, a - m, b - m, c - m));
        }
        if (lane == 0) out[d.at(q.x, q.y, q.z)] = !beaten;
    }
}

// dd, kernels_no_3d_write.cl:970-1004 (in-range voxels only): of every cell's
// candidates the one with the greatest TDF above 0, of equal ones the first in
// x, y, z order (z innermost).  A workgroup takes whole cells of one (y, z)
// row of cells: a thread finds the best of each of its V columns (rows of the
// mask are read as they lie, V bytes a thread and access, eight accesses in
// flight), then the first column of a cell takes the best of its columns in x
// order.  V = 4 where rows are whole words.  Candidates are few, so the mask's
// bytes bound it: 400 x 512 x 512, cube 5: 124 us with a thread per cell, 170
// with V = 1, 59 with V = 4.
constexpr int CM_T = 128;
template <int V>
__global__ void __launch_bounds__(CM_T) k_cube_max(const float* __restrict__ tdf, const uint8_t* __restrict__ cand,
                                                   Dims d, int cube, int cols, uint8_t* __restrict__ out) {
    __shared__ float top[CM_T * V];
    __shared__ int at[CM_T * V];  // z * cube + y within the cell
    const int xl = threadIdx.x * V, x0 = blockIdx.x * cols, x = x0 + xl;
    const int y0 = blockIdx.y * cube, z0 = blockIdx.z * cube;
    float best[V];
    int bi[V];
#pragma unroll
    for (int e = 0; e < V; e++) {
        best[e] = 0.0f;
        bi[e] = -1;
    }
    if (xl < cols && x < d.X) {
        const int ny = min(cube, d.Y - y0), nz = min(cube, d.Z - z0), n = ny * nz;
        int b = 0, c = 0;
        for (int j = 0; j < n; j += 8) {
            i64 i[8];
            unsigned m[8];
            int q[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                q[k] = c * cube + b;
                i[k] = d.at(x, y0 + b, z0 + c);
                m[k] = V == 4 ? *reinterpret_cast<const unsigned*>(cand + i[k]) : cand[i[k]];
                if (j + k >= n) m[k] = 0;  // a repeat of the last voxel
                c++;
                if (c == nz) {
                    c = b + 1 < ny ? 0 : nz - 1;
                    b = b + 1 < ny ? b + 1 : b;
                }
            }
#pragma unroll
            for (int k = 0; k < 8; k++) {
                if (m[k] == 0) continue;
#pragma unroll
                for (int e = 0; e < V; e++)
                    if (((m[k] >> (8 * e)) & 0xffu) == 1u) {
                        const float t = tdf[i[k] + e];
                        if (t > best[e]) {
                            best[e] = t;
                            bi[e] = q[k];
                        }
                    }
            }
        }
    }
#pragma unroll
    for (int e = 0; e < V; e++) {
        top[xl + e] = best[e];
        at[xl + e] = bi[e];
    }
    __syncthreads();
    for (int l = threadIdx.x * cube; l < cols && x0 + l < d.X; l += CM_T * cube) {
        float m = 0.0f;
        int k = -1;
        for (int a = l; a < l + cube; a++)
            if (top[a] > m) {
                m = top[a];
                k = a;
            }
        if (k >= 0) out[d.at(x0 + k, y0 + at[k] % cube, z0 + at[k] / cube)] = 1;
    }
}

}  // namespace tsf

using namespace tsf;

extern "C" {

tsf_status tsf_hessian_eigen(const tsf_field* field, tsf_dims dims, int32_t normalize, float* lambda, float* vectors,
                             hipStream_t stream) {
    const char* W = "tsf_hessian_eigen";
    TSF_TRY(check_field(field, normalize != 0, W));
    TSF_TRY(check_dims(dims, 1, W));
    if (!lambda) return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: NULL lambda", W);
    Dims d = D(dims);
    dim3 grid((d.X + 63) / 64, (d.Y + 3) / 4, d.Z), block(64, 4);
    const float inv = 1.0f / field->scale;
    switch (field->storage) {
        case TSF_STORAGE_F32: {
            Field<F32> F{(const float*)field->x, (const float*)field->y, (const float*)field->z, (const float*)field->w, inv};
            if (normalize) hipLaunchKernelGGL((k_hessian_eigen<F32, true>), grid, block, 0, stream, F, d, lambda, vectors);
            else hipLaunchKernelGGL((k_hessian_eigen<F32, false>), grid, block, 0, stream, F, d, lambda, vectors);
            break;
        }
        case TSF_STORAGE_F16: {
            typedef __half T;
            Field<F16> F{(const T*)field->x, (const T*)field->y, (const T*)field->z, (const T*)field->w, inv};
            if (normalize) hipLaunchKernelGGL((k_hessian_eigen<F16, true>), grid, block, 0, stream, F, d, lambda, vectors);
            else hipLaunchKernelGGL((k_hessian_eigen<F16, false>), grid, block, 0, stream, F, d, lambda, vectors);
            break;
        }
        case TSF_STORAGE_SN16: {
            typedef short T;
            Field<SN16> F{(const T*)field->x, (const T*)field->y, (const T*)field->z, (const T*)field->w, inv};
            if (normalize) hipLaunchKernelGGL((k_hessian_eigen<SN16, true>), grid, block, 0, stream, F, d, lambda, vectors);
            else hipLaunchKernelGGL((k_hessian_eigen<SN16, false>), grid, block, 0, stream, F, d, lambda, vectors);
            break;
        }
        default: {
            typedef __hip_bfloat16 T;
            Field<BF16> F{(const T*)field->x, (const T*)field->y, (const T*)field->z, (const T*)field->w, inv};
            if (normalize) hipLaunchKernelGGL((k_hessian_eigen<BF16, true>), grid, block, 0, stream, F, d, lambda, vectors);
            else hipLaunchKernelGGL((k_hessian_eigen<BF16, false>), grid, block, 0, stream, F, d, lambda, vectors);
        }
    }
    return check_launch(W);
}

tsf_status tsf_do_eigen_points(const float* fx, const float* fy, const float* fz, tsf_dims dims,
                               const int32_t* positions, int64_t count, float* out, hipStream_t stream) {
    const char* W = "tsf_do_eigen_points";
    if (!fx || !fy || !fz || !out || (count > 0 && !positions))
        return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: NULL argument", W);
    TSF_TRY(check_dims(dims, 3, W));
    if (count < 0) return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: negative count", W);
    if (count == 0) return TSF_OK;
    hipLaunchKernelGGL(k_do_eigen_points, (unsigned)((count + 255) / 256), 256, 0, stream, fx, fy, fz, D(dims),
                       positions, (i64)count, out);
    return check_launch(W);
}

tsf_status tsf_candidate_nms(const float* tdf, const float* radius, const tsf_field* field, tsf_dims dims,
                             const int32_t* positions, int64_t count, int32_t maxd_cap, uint8_t* out,
                             hipStream_t stream) {
    const char* W = "tsf_candidate_nms";
    (void)tdf;
    TSF_TRY(check_field(field, true, W));
    TSF_TRY(check_dims(dims, 1, W));
    if (!radius || !out || (count > 0 && !positions))
        return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: NULL argument", W);
    if (maxd_cap < 1 || maxd_cap > 64) return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: maxd_cap out of [1, 64]", W);
    if (count < 0) return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: negative count", W);
    if (count == 0) return TSF_OK;
    Dims d = D(dims);
    const float inv = 1.0f / field->scale;
    unsigned g = (unsigned)((count + 255) / 256);
    switch (field->storage) {
        case TSF_STORAGE_F32: {
            Field<F32> F{(const float*)field->x, (const float*)field->y, (const float*)field->z, (const float*)field->w, inv};
            hipLaunchKernelGGL(k_candidate_nms<F32>, g, 256, 0, stream, radius, F, d, positions, (i64)count, maxd_cap, out);
            break;
        }
        case TSF_STORAGE_F16: {
            typedef __half T;
            Field<F16> F{(const T*)field->x, (const T*)field->y, (const T*)field->z, (const T*)field->w, inv};
            hipLaunchKernelGGL(k_candidate_nms<F16>, g, 256, 0, stream, radius, F, d, positions, (i64)count, maxd_cap, out);
            break;
        }
        case TSF_STORAGE_SN16: {
            typedef short T;
            Field<SN16> F{(const T*)field->x, (const T*)field->y, (const T*)field->z, (const T*)field->w, inv};
            hipLaunchKernelGGL(k_candidate_nms<SN16>, g, 256, 0, stream, radius, F, d, positions, (i64)count, maxd_cap, out);
            break;
        }
        default: {
            typedef __hip_bfloat16 T;
            Field<BF16> F{(const T*)field->x, (const T*)field->y, (const T*)field->z, (const T*)field->w, inv};
            hipLaunchKernelGGL(k_candidate_nms<BF16>, g, 256, 0, stream, radius, F, d, positions, (i64)count, maxd_cap, out);
        }
    }
    return check_launch(W);
}

tsf_status tsf_cube_max(const float* tdf, const uint8_t* candidates, tsf_dims dims, int32_t cube, uint8_t* out,
                        hipStream_t stream) {
    const char* W = "tsf_cube_max";
    if (!tdf || !candidates || !out) return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: NULL argument", W);
    TSF_TRY(check_dims(dims, 1, W));
    if (cube < 1 || cube > 64) return set_error(TSF_ERR_INVALID_ARGUMENT, "%s: cube size out of [1, 64]", W);
    Dims d = D(dims);
    const bool words = d.X % 4 == 0 && (uintptr_t)candidates % 4 == 0;
    const int unit = words ? 4 * cube : cube, cols = (words ? 4 : 1) * CM_T / unit * unit;  // whole cells and words
    const dim3 grid((d.X + cols - 1) / cols, (d.Y + cube - 1) / cube, (d.Z + cube - 1) / cube);
    if (words)
        hipLaunchKernelGGL(k_cube_max<4>, grid, CM_T, 0, stream, tdf, candidates, d, cube, cols, out);
    else
        hipLaunchKernelGGL(k_cube_max<1>, grid, CM_T, 0, stream, tdf, candidates, d, cube, cols, out);
    return check_launch(W);
}

}  // extern "C"
