// RMSNorm of training (chassis.py:96-106) on bf16 rows with a float32 weight:
//     r = rsqrt(mean(x^2) + eps),  xn = bf16(x r),  y = xn w   (float32)
// and its backward
//     g = bf16(gy w),  gx = bf16(r g - x r^3 mean(g x)),  gw = sum_rows gy xn
// with the roundings of the element-by-element form.  A wavefront takes a row
// at a time (a lane 4 columns of every 256); the weight gradient is summed
// per lane over the workgroup's rows, then over workgroups by a second kernel
// in a fixed order.  Bound by memory: 8,192 x 512, forward 29 MB in 8 us,
// backward 34 MB in 14 us plus 5 us for the sum; as nine and twenty-two
// elementwise kernels they took 60 and 135 us.
#include "common.h"

namespace walsh {

constexpr int kNormWaves = 4;
constexpr int kNormMaxC = 2048;

__device__ __forceinline__ float norm_sum(float v) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
    return v;
}
__device__ __forceinline__ f32x4 round_bf16(f32x4 v) {
    const uint32_t a = pack_bf16x2(v.x, v.y), b = pack_bf16x2(v.z, v.w);
    return f32x4{__uint_as_float(a << 16), __uint_as_float(a & 0xffff0000u), __uint_as_float(b << 16),
                 __uint_as_float(b & 0xffff0000u)};
}

// K: 256-column pieces of a row.
template <int K>
__global__ __launch_bounds__(64 * kNormWaves) void rmsnorm_fwd_kernel(const uint16_t *__restrict__ x,
                                                                      const float *__restrict__ w, int64_t M, int C,
                                                                      float eps, float *__restrict__ y,
                                                                      float *__restrict__ rstd) {
    const int lane = threadIdx.x & 63;
    f32x4 wv[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int c = 256 * k + 4 * lane;
        wv[k] = c < C ? load4(w + c) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int64_t t = (int64_t)blockIdx.x * kNormWaves + (threadIdx.x >> 6); t < M;
         t += (int64_t)gridDim.x * kNormWaves) {
        f32x4 xv[K];
        float ss = 0.f;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = 256 * k + 4 * lane;
            xv[k] = c < C ? load4(x + t * C + c) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int k = 0; k < K; ++k) ss += xv[k].x * xv[k].x + xv[k].y * xv[k].y + xv[k].z * xv[k].z + xv[k].w * xv[k].w;
        const float r = rsqrtf(norm_sum(ss) / (float)C + eps);
        if (lane == 0) rstd[t] = r;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = 256 * k + 4 * lane;
            if (c < C) store4(y + t * C + c, round_bf16(xv[k] * r) * wv[k]);
        }
    }
}

template <int K>
__global__ __launch_bounds__(64 * kNormWaves) void rmsnorm_bwd_kernel(const uint16_t *__restrict__ x,
                                                                      const float *__restrict__ w,
                                                                      const float *__restrict__ rstd,
                                                                      const float *__restrict__ gy, int64_t M, int C,
                                                                      uint16_t *__restrict__ gx,
                                                                      float *__restrict__ parts) {
    __shared__ f32x4 sum[kNormWaves - 1][K * 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    f32x4 wv[K], gw[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int c = 256 * k + 4 * lane;
        wv[k] = gx && c < C ? load4(w + c) : f32x4{0.f, 0.f, 0.f, 0.f};
        gw[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int64_t t = (int64_t)blockIdx.x * kNormWaves + wave; t < M; t += (int64_t)gridDim.x * kNormWaves) {
        f32x4 xv[K], g[K];
        const float r = rstd[t];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = 256 * k + 4 * lane;
            xv[k] = c < C ? load4(x + t * C + c) : f32x4{0.f, 0.f, 0.f, 0.f};
            g[k] = c < C ? load4(gy + t * C + c) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
        float dot = 0.f;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            gw[k] += g[k] * round_bf16(xv[k] * r);
            g[k] = round_bf16(g[k] * wv[k]);
            dot += g[k].x * xv[k].x + g[k].y * xv[k].y + g[k].z * xv[k].z + g[k].w * xv[k].w;
        }
        if (!gx) continue;
        const float f = norm_sum(dot) * (r * r * r) / (float)C;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int c = 256 * k + 4 * lane;
            if (c < C) store4(gx + t * C + c, g[k] * r - xv[k] * f);
        }
    }
    if (!parts) return;
    if (wave > 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) sum[wave - 1][k * 64 + lane] = gw[k];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int c = 256 * k + 4 * lane;
#pragma unroll
        for (int v = 0; v < kNormWaves - 1; ++v) gw[k] += sum[v][k * 64 + lane];
        if (c < C) store4(parts + (int64_t)blockIdx.x * C + c, gw[k]);
    }
}

// gw[c] = sum of the G workgroups' partial sums: 64 columns per workgroup, 16
// wavefronts taking every 16th row.
__global__ __launch_bounds__(1024) void rmsnorm_sum_kernel(const float *__restrict__ parts, int G, int C,
                                                           float *__restrict__ gw) {
    __shared__ float sum[16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = blockIdx.x * 64 + lane;
    float acc = 0.f;
    if (c < C) {
#pragma unroll 8
        for (int g = wave; g < G; g += 16) acc += parts[(int64_t)g * C + c];
    }
    sum[wave][lane] = acc;
    __syncthreads();
    if (wave > 0 || c >= C) return;
#pragma unroll
    for (int v = 1; v < 16; ++v) acc += sum[v][lane];
    gw[c] = acc;
}

static int64_t norm_grid(int64_t M) {
    const int64_t g = ceil_div(M, 2 * kNormWaves), most = 2 * (int64_t)device_info().cu_count;
    return g < most ? g : most;
}

static int norm_check(const char *fn, int64_t M, int64_t C, const void *x, const void *w, const void *y) {
    if (M < 1 || C < 4 || C % 4 || C > kNormMaxC)
        return set_error(WALSH_ENOTSUP, "%s: needs M >= 1 and C <= 2048, a multiple of 4 (M=%lld C=%lld)", fn,
                         (long long)M, (long long)C);
    if ((uintptr_t)x % 8 || (uintptr_t)w % 16 || (uintptr_t)y % 16)
        return set_error(WALSH_EINVAL, "%s: rows of x 8-byte, float rows 16-byte aligned", fn);
    return WALSH_OK;
}

}  // namespace walsh

using namespace walsh;

WALSH_EXPORT int walsh_rmsnorm_fwd(const void *x, const float *w, int64_t M, int64_t C, float eps, float *y, float *rstd,
                                   void *stream) {
    const char *fn = "walsh_rmsnorm_fwd";
    if (!x || !w || !y || !rstd) return set_error(WALSH_EINVAL, "%s: null pointer", fn);
    const int rc = norm_check(fn, M, C, x, w, y);
    if (rc) return rc;
    const int64_t rows = ceil_div(M, kNormWaves), most = 8 * (int64_t)device_info().cu_count;
    const dim3 G((unsigned)(rows < most ? rows : most)), B(64 * kNormWaves);
    auto go = [&](auto kernel) {
        launch(kernel, G, B, 0, (hipStream_t)stream, (const uint16_t *)x, w, M, (int)C, eps, y, rstd);
    };
    if (C <= 256) go(rmsnorm_fwd_kernel<1>);
    else if (C <= 512) go(rmsnorm_fwd_kernel<2>);
    else if (C <= 1024) go(rmsnorm_fwd_kernel<4>);
    else go(rmsnorm_fwd_kernel<8>);
    return check_hip(hipGetLastError(), fn);
}

WALSH_EXPORT int64_t walsh_rmsnorm_bwd_workspace_bytes(int64_t M, int64_t C) {
    return M < 1 || C < 1 ? 0 : norm_grid(M) * C * 4;
}

WALSH_EXPORT int walsh_rmsnorm_bwd(const void *x, const float *w, const float *rstd, const float *gy, int64_t M,
                                   int64_t C, void *gx, float *gw, void *work, int64_t work_bytes, void *stream) {
    const char *fn = "walsh_rmsnorm_bwd";
    if (!x || (gx && !w) || !rstd || !gy || (gw && !work)) return set_error(WALSH_EINVAL, "%s: null pointer", fn);
    int rc = norm_check(fn, M, C, x, w, gy);
    if (rc) return rc;
    if (!gx && !gw) return WALSH_OK;
    if ((uintptr_t)gx % 8 || (gw && (work_bytes < walsh_rmsnorm_bwd_workspace_bytes(M, C) || (uintptr_t)work % 16)))
        return set_error(WALSH_EINVAL, "%s: gx 8-byte aligned; workspace of %lld bytes (16-aligned), needs %lld", fn,
                         (long long)work_bytes, (long long)walsh_rmsnorm_bwd_workspace_bytes(M, C));
    const int64_t grid = norm_grid(M);
    float *parts = gw ? (float *)work : nullptr;
    auto go = [&](auto kernel) {
        launch(kernel, dim3((unsigned)grid), dim3(64 * kNormWaves), 0, (hipStream_t)stream, (const uint16_t *)x, w, rstd,
               gy, M, (int)C, (uint16_t *)gx, parts);
    };
    if (C <= 256) go(rmsnorm_bwd_kernel<1>);
    else if (C <= 512) go(rmsnorm_bwd_kernel<2>);
    else if (C <= 1024) go(rmsnorm_bwd_kernel<4>);
    else go(rmsnorm_bwd_kernel<8>);
    rc = check_hip(hipGetLastError(), fn);
    if (rc || !gw) return rc;
    launch(rmsnorm_sum_kernel, dim3((unsigned)ceil_div(C, 64)), dim3(1024), 0, (hipStream_t)stream, (const float *)parts,
           (int)grid, (int)C, gw);
    return check_hip(hipGetLastError(), fn);
}
