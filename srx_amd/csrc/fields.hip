// fields.hip -- conversion of the device state to the caller's layout: fields leave the GPU as the
// reference lays them out (per voxel, 3x3 row-major tensors or 12 values per slip system), spectra
// as the FFT entry points return them.
#include "kern_common.hpp"

namespace srx {

// One chunk of a field, voxels [v0, v0 + nv), from component-major state to nc values per voxel at
// `out`, which srx_get_field points at pinned host memory: the kernel's stores cross PCIe directly.
// Bound by that link; a block turns its 256 voxels around in LDS so that every wavefront's store is one
// contiguous run of 512 B (54 GB/s measured into 2 MiB of pinned memory, against 3-4 GB/s for copying
// the components to pageable memory and interleaving them there: the stress of 128^3, 151 MB, took
// 57 ms).  The arithmetic is the host formulas' own, without contraction.
constexpr int GATHER_BLOCK = 256;
template <int MODE, int NC>
__global__ void __launch_bounds__(GATHER_BLOCK) k_gather(FieldSrc src, int v0, int nv, double *__restrict__ out) {
#pragma clang fp contract(off)
    __shared__ double buf[GATHER_BLOCK * NC];
    const int b0 = blockIdx.x * GATHER_BLOCK, cnt = min(GATHER_BLOCK, nv - b0);
    if ((int)threadIdx.x < cnt) {
        const size_t v = (size_t)v0 + b0 + threadIdx.x, N = src.n;
        double *o = buf + threadIdx.x * NC;
        if constexpr (MODE == FIELD_INT) {
            o[0] = (double)src.i[v];
        } else if constexpr (MODE == FIELD_B6) {
            double b6[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) b6[k] = k < src.comps ? src.a[k * N + v] : 0.0;
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    double s = 0.0;
#pragma unroll
                    for (int k = 0; k < 6; ++k) s += b6[k] * bbasis(k, r, c);
                    o[3 * r + c] = s;
                }
        } else {
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                double x = src.a[k * N + v];
                if constexpr (MODE == FIELD_RATE) x = (x - src.b[k * N + v]) / src.dt;
                if constexpr (MODE == FIELD_FLUCT) x = (x - src.u[k]) + (src.b ? src.b[k * N + v] : 0.0);
                o[k] = x;
            }
        }
    }
    __syncthreads();
    double *dst = out + (size_t)b0 * NC;
    for (int i = threadIdx.x; i < cnt * NC; i += GATHER_BLOCK) dst[i] = buf[i];
}

hipError_t launch_gather(hipStream_t s, int mode, int nc, const FieldSrc &src, int v0, int nv, double *out) {
    const dim3 g((nv + GATHER_BLOCK - 1) / GATHER_BLOCK), b(GATHER_BLOCK);
    switch (mode) {
    case FIELD_INT: hipLaunchKernelGGL((k_gather<FIELD_INT, 1>), g, b, 0, s, src, v0, nv, out); break;
    case FIELD_B6: hipLaunchKernelGGL((k_gather<FIELD_B6, 9>), g, b, 0, s, src, v0, nv, out); break;
    case FIELD_RATE: hipLaunchKernelGGL((k_gather<FIELD_RATE, 9>), g, b, 0, s, src, v0, nv, out); break;
    case FIELD_FLUCT: hipLaunchKernelGGL((k_gather<FIELD_FLUCT, 9>), g, b, 0, s, src, v0, nv, out); break;
    default:
        if (nc == 12) hipLaunchKernelGGL((k_gather<FIELD_PLAIN, 12>), g, b, 0, s, src, v0, nv, out);
        else if (nc == 9) hipLaunchKernelGGL((k_gather<FIELD_PLAIN, 9>), g, b, 0, s, src, v0, nv, out);
        else hipLaunchKernelGGL((k_gather<FIELD_PLAIN, 1>), g, b, 0, s, src, v0, nv, out);
    }
    return check_launch("gather");
}

// Spectra between the passes' layout C [c][kz][y][x] (complex T) and the entry points' [c][x][y][kz]
// (complex double).  Bound by memory: for every (c, y) a block turns a TILE x TILE piece around in LDS,
// so that both sides move in runs of 512 B (half of it for complex T = float).  The same reordering in
// strided loops on the host was most of srx_fft_forward and srx_fft_inverse: 9.2 ms for both with 6 fields
// of 60 x 64 x 75, 4.0 ms with this kernel, most of it the copies over PCIe.
constexpr int TURN_TILE = 32, TURN_BLOCK = 256;
template <typename T, bool OUT>
__global__ void __launch_bounds__(TURN_BLOCK) k_spec_turn(T *__restrict__ spec, double *__restrict__ user, int n0, int n1,
                                                          int H) {
    typedef T T2 __attribute__((ext_vector_type(2)));
    // the caller's buffer may be aligned to 8 bytes only
    typedef double U2 __attribute__((ext_vector_type(2), aligned(8)));
    __shared__ U2 tile[TURN_TILE][TURN_TILE + 1];   // [x][kz]
    const int c = blockIdx.z / n1, y = blockIdx.z % n1;
    const int x0 = blockIdx.x * TURN_TILE, k0 = blockIdx.y * TURN_TILE;
    const int i = threadIdx.x % TURN_TILE;
    T2 *sp = reinterpret_cast<T2 *>(spec);
    U2 *us = reinterpret_cast<U2 *>(user);
    auto at_spec = [&](int x, int kz) { return (((size_t)c * H + kz) * n1 + y) * n0 + x; };
    auto at_user = [&](int x, int kz) { return (((size_t)c * n0 + x) * n1 + y) * H + kz; };
#pragma unroll
    for (int j = threadIdx.x / TURN_TILE; j < TURN_TILE; j += TURN_BLOCK / TURN_TILE) {
        if (OUT && x0 + i < n0 && k0 + j < H) {
            const T2 v = sp[at_spec(x0 + i, k0 + j)];
            tile[i][j] = U2{(double)v.x, (double)v.y};
        } else if (!OUT && x0 + j < n0 && k0 + i < H) {
            tile[j][i] = us[at_user(x0 + j, k0 + i)];
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = threadIdx.x / TURN_TILE; j < TURN_TILE; j += TURN_BLOCK / TURN_TILE) {
        if (OUT && x0 + j < n0 && k0 + i < H) {
            us[at_user(x0 + j, k0 + i)] = tile[j][i];
        } else if (!OUT && x0 + i < n0 && k0 + j < H) {
            const U2 v = tile[i][j];
            T2 o;
            o.x = (T)v.x;
            o.y = (T)v.y;
            sp[at_spec(x0 + i, k0 + j)] = o;
        }
    }
}

hipError_t launch_spec_turn(hipStream_t s, int prec, bool out, void *spec, double *user, int ncomp, const int n[3]) {
    const int H = n[2] / 2 + 1;
    const dim3 g((n[0] + TURN_TILE - 1) / TURN_TILE, (H + TURN_TILE - 1) / TURN_TILE, ncomp * n[1]), b(TURN_BLOCK);
    if (prec != 0) {
        if (out) hipLaunchKernelGGL((k_spec_turn<float, true>), g, b, 0, s, (float *)spec, user, n[0], n[1], H);
        else hipLaunchKernelGGL((k_spec_turn<float, false>), g, b, 0, s, (float *)spec, user, n[0], n[1], H);
    } else {
        if (out) hipLaunchKernelGGL((k_spec_turn<double, true>), g, b, 0, s, (double *)spec, user, n[0], n[1], H);
        else hipLaunchKernelGGL((k_spec_turn<double, false>), g, b, 0, s, (double *)spec, user, n[0], n[1], H);
    }
    return check_launch("spec_turn");
}

}  // namespace srx
